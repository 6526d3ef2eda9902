"""Benchmark: XAS spectra/s of a parameter-fitting loop on one MI355X --
batched exact diagonalization plus the learned surrogate, against plain
(unbatched) GPU ED, at L1 error <= 1e-2.

Default workload ("fit"), one step = one iteration of a 256-walker
Metropolis fitting loop over the 8 parameters (10Dq, F0, F2/F4 scale, charge
transfer, V_eg, V_t2g, xi_3d, T) of a NiO-like 10-bath impurity model: every
walker proposes a move and needs the thermal, polarization-summed L2,3 XAS of
its proposal (3 lowest eigenstates, energy cut, 3 dipole polarizations,
200-step Lanczos, continued fraction on 1000 points, complex128).  Proposals
the ensemble agrees on are answered by the surrogate network at once; the
others wait and are evaluated together by one batched exact-ED call once
half the walkers wait (and at the end of the timed steps), so the timed
region contains every proposal's spectrum.  Set-up (untimed, reported): a 20k-spectrum
training set from the batched exact ED (the configuration's size), 5-member ensemble training with the
library's BF16 matrix-core kernels, trust-threshold calibration on 2048
validation spectra.  After the timed steps every surrogate-served spectrum
is recomputed by exact ED and its L1 error reported.  The same loop without
the surrogate gives the batched-ED rate, and per-model unbatched runs of
the same proposals give the plain GPU ED rate.

``--workload batched128``: 128 seeded models with bath sizes 10-50 (26-66
spin-orbitals) per step, exact path only (the batched-ED configuration).
``--workload exact``: the fitting family's batched exact-ED call alone
(``--models`` proposals per call), no surrogate and no training.

The timed loops run as the product does, without kernel timing; each is
then repeated with the same seeds (the same walk) with a HIP-event pair
around every kernel launch, which gives the kernels' average durations.
A trusted proposal's misfit is computed on the device, so the served
spectra stay there during the loop; they are predicted again for scoring
(a sample's row does not depend on the rest of its batch).

Prints one JSON line with a roofline figure for the dominant kernel
(from the instrumented repeat) and a CPU baseline: the oracle (a
pure Python/numpy restatement of the reference algorithm) on a bounded
sample of the same spectra, one model per worker process.
"""

import argparse
import json
import multiprocessing as mp
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "XAS spectra/s on 1 MI355X: batched+surrogate vs plain GPU ED @ L1 err≤1e-2"
HBM_PEAK_GBS = 8000.0


def algorithmic_bytes_lanczos(n, nnz, k):
    """20 nnz + 4(n+1) + 48 n bytes per Lanczos step (complex128 values,
    int32 columns/rowptr, read v_j, v_{j-1}, write w)."""
    n = np.asarray(n, np.float64)
    nnz = np.asarray(nnz, np.float64)
    k = np.asarray(k, np.float64)
    return float(np.sum(k * (20 * nnz + 4 * (n + 1) + 48 * n)))


def algorithmic_bytes_eigen(n, nnz, steps):
    """HBM bytes of the eigensolver's Lanczos steps, priced like any Lanczos
    step: per chain, steps x (20 nnz + 4(n+1) + 48 n).  The Gram-Schmidt
    passes over the stored Krylov vectors are not counted: for the
    few-hundred-state sectors of these workloads the vectors sit in LDS and
    L2, not in HBM (see ``gram_schmidt_bytes``)."""
    return algorithmic_bytes_lanczos(n, nnz, steps)


def eigen_itemsize(fam):
    """Bytes per Krylov-vector element of the family's eigensolver: 8 when
    every Hamiltonian coefficient is real (the real kernel), else 16."""
    return 8 if not (np.any(fam.c0.imag) or np.any(fam.cmat.imag)) else 16


def gram_schmidt_bytes(n, steps, itemsize=16):
    """On-chip bytes the eigensolver's classical Gram-Schmidt reads: at step j
    the j stored vectors are read twice (dots, update), one pass: 2 j n
    itemsize summed over the steps.  Reported as a work rate, not HBM."""
    tot = 0.0
    for ni, si in zip(n, steps):
        s = float(si)
        tot += 2.0 * itemsize * float(ni) * s * (s + 1) / 2
    return tot


# ------------------------------------------------------------------ CPU baseline (oracle)


def _oracle_batched(args):
    """One batched-workload model's XAS with the CPU oracle (reference algorithm)."""
    p, omega, K = args
    sys.path.insert(0, ROOT)
    from impuritymodel_amd.models import model_from_params
    from impuritymodel_amd.operators import getDipoleOperators
    from oracle import basis, krylov, spectra

    m = model_from_params(p)
    n = m.n_spin_orbitals
    b = basis.get_basis(m.nBaths, m.nValBaths, m.dnValBaths, m.dnConBaths, m.dnTols, m.n0imps)
    es, psis = krylov.eigensystem(n, m.hOp, b, 3, eigenValueTol=1e-12)
    es = spectra.energy_cut(tuple(es))
    tops = getDipoleOperators(m.nBaths, ([1, 0, 0], [0, 1, 0], [0, 0, 1]))
    _, _, s = spectra.xas(n, m.hOp, tops, psis[: len(es)], es, omega, 0.2, m.restrictions, krylovSize=K)
    return s


def _oracle_family(theta):
    """One fitting-loop spectrum with the CPU oracle."""
    sys.path.insert(0, ROOT)
    from impuritymodel_amd import surrogate as S
    from impuritymodel_amd.operators import getDipoleOperators
    from oracle import basis, krylov, spectra

    fam = S.XASFamily()
    m = fam.models(np.asarray([theta]))[0]
    n = m.n_spin_orbitals
    b = basis.get_basis(m.nBaths, m.nValBaths, m.dnValBaths, m.dnConBaths, m.dnTols, m.n0imps)
    es, psis = krylov.eigensystem(n, m.hOp, b, 3, eigenValueTol=1e-12)
    es = spectra.energy_cut(tuple(es), T=theta[7])
    tops = getDipoleOperators(m.nBaths, ([1, 0, 0], [0, 1, 0], [0, 0, 1]))
    _, _, s = spectra.xas(n, m.hOp, tops, psis[: len(es)], es, S.OMEGA, S.DELTA, m.restrictions, T=theta[7],
                          krylovSize=200)
    return s


def _warm(_):
    """Worker warm-up: the imports and first-call set-up of a spectrum."""
    sys.path.insert(0, ROOT)
    import scipy.sparse.linalg  # noqa: F401

    from impuritymodel_amd import surrogate  # noqa: F401
    from oracle import basis, krylov, spectra  # noqa: F401

    return os.getpid()


def cpu_baseline(fn, items, workers, what, per_worker=4):
    """Oracle spectra/s on a bounded sample: ``per_worker`` spectra for each of
    ``workers`` processes, timed after the pool has started and every worker
    has imported the oracle and computed one untimed spectrum."""
    sample = items[: workers * per_worker]
    ctx = mp.get_context("spawn")
    with ctx.Pool(workers) as pool:
        pool.map(_warm, range(workers), chunksize=1)
        pool.map(fn, items[-workers:], chunksize=1)  # one untimed spectrum per worker
        t0 = time.perf_counter()
        pool.map(fn, sample, chunksize=per_worker)
        dt = time.perf_counter() - t0
    return dict(value=round(len(sample) / dt, 4), unit="spectra/s", cores=workers, kind="port",
                sample="%d %s on %d warm worker processes (%d each), %.1f s wall, start-up excluded"
                       % (len(sample), what, workers, per_worker, dt))


def measured_peaks(torch):
    """HBM copy bandwidth and dense bf16 GEMM rate measured on this GPU
    (reported next to the nominal 8 TB/s and 2.5 PFLOP/s)."""
    out = {}
    n = 1 << 28  # 1 GiB of float32 each way
    src = torch.ones(n, dtype=torch.float32, device="cuda")
    dst = torch.empty_like(src)
    for _ in range(3):
        dst.copy_(src)
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    reps = 20
    for _ in range(reps):
        dst.copy_(src)
    e1.record()
    torch.cuda.synchronize()
    out["copy_gbs"] = round(reps * 2 * 4 * n / (e0.elapsed_time(e1) * 1e-3) / 1e9, 1)
    del src, dst
    m = 8192
    a = torch.randn(m, m, dtype=torch.bfloat16, device="cuda")
    b = torch.randn(m, m, dtype=torch.bfloat16, device="cuda")
    for _ in range(3):
        torch.matmul(a, b)
    torch.cuda.synchronize()
    e0.record()
    reps = 20
    for _ in range(reps):
        torch.matmul(a, b)
    e1.record()
    torch.cuda.synchronize()
    out["bf16_gemm_tflops"] = round(reps * 2.0 * m ** 3 / (e0.elapsed_time(e1) * 1e-3) / 1e12, 1)
    out["how"] = "1 GiB device copy (read + write bytes) and an 8192^3 bf16 matmul, torch on the engine's GPU"
    del a, b
    torch.cuda.empty_cache()
    return out


BF16_MFMA_PEAK_TFLOPS = 2500.0  # dense bf16 matrix-core peak of one MI355X


def _pmc_traffic(kernel, workload=None):
    """HBM bytes per dispatch of ``kernel`` measured by the rocprofv3 --pmc
    runs (FETCH_SIZE + WRITE_SIZE, calibrated against a copy of known size)
    whose summaries are kept in profiles/, or None.  A line tagged with a
    workload (``workload=...``) counts only for that workload."""
    import glob
    import re

    for path in sorted(glob.glob(os.path.join(ROOT, "profiles", "*pmc_traffic.md"))):
        with open(path) as f:
            for line in f:
                m = re.match(r"traffic_bytes_per_dispatch kernel=(\S+) bytes=(\d+)(?: workload=(\S+))?", line.strip())
                if m and m.group(1) == kernel and (m.group(3) is None or m.group(3) == workload):
                    return int(m.group(2))
    return None


def _tuning_value(args, name, default):
    """The value ``--tuning name=value`` set for this run, or the engine's default."""
    for kv in getattr(args, "tuning", []) or []:
        k, v = kv.split("=", 1)
        if k == name:
            return int(v)
    return default


# the kernel behind a launch class, where its name is another (chains of the
# fitting family run on the register kernels, every surrogate product on one GEMM)
KERNEL_NAMES = {"eigen": "eigen_reg_kernel", "lanczos": "lanczos_reg_kernel", "mlp_gemm": "gemm_nt_kernel",
                "mlp_adam": "gemm_nt_kernel"}


def _roofline(kernels, bytes_by_kernel, flops_by_kernel=None, workload=None, names=KERNEL_NAMES):
    """Roofline object of the kernel with the largest timed total: HBM-bound
    kernels priced by algorithmic bytes against 8 TB/s, matrix-core kernels
    by algorithmic flops against the dense bf16 peak."""
    flops_by_kernel = flops_by_kernel or {}
    cand = {k: v for k, v in kernels.items() if (k in bytes_by_kernel or k in flops_by_kernel) and v[1] > 0}
    if not cand:
        return None
    dom = max(cand, key=lambda k: cand[k][0])
    ms_total, launches = cand[dom]
    avg_ms = ms_total / launches
    name = names.get(dom, dom + "_kernel")
    if dom in flops_by_kernel:
        per_launch = flops_by_kernel[dom] / launches
        achieved = per_launch / (avg_ms * 1e-3) / 1e12
        return dict(bound="mfma", kernel=name, achieved=round(achieved, 3), peak=BF16_MFMA_PEAK_TFLOPS,
                    unit="TFLOP/s", frac=round(achieved / BF16_MFMA_PEAK_TFLOPS, 5), traffic=_pmc_traffic(name, workload),
                    avg_launch_ms=round(avg_ms, 4), launches=launches, algorithmic_flops_per_launch=per_launch)
    per_launch = bytes_by_kernel[dom] / launches
    achieved = per_launch / (avg_ms * 1e-3) / 1e9
    return dict(bound="hbm", kernel=name, achieved=round(achieved, 2), peak=HBM_PEAK_GBS, unit="GB/s",
                frac=round(achieved / HBM_PEAK_GBS, 4), traffic=_pmc_traffic(name, workload), avg_launch_ms=round(avg_ms, 4),
                launches=launches, algorithmic_bytes_per_launch=per_launch)


KERNELS = ("eigen", "lanczos", "apply_count", "apply_fill", "cf", "mlp_gemm", "mlp_adam")


class _Roctx:
    """roctx ranges around the timed regions (seen by rocprofv3 --marker-trace); no-ops without the library."""

    def __init__(self):
        import ctypes

        try:
            self.lib = ctypes.CDLL("librocprofiler-sdk-roctx.so")
            self.lib.roctxRangePushA.argtypes = [ctypes.c_char_p]
        except OSError:
            self.lib = None

    def push(self, name):
        if self.lib is not None:
            self.lib.roctxRangePushA(name.encode())

    def pop(self):
        if self.lib is not None:
            self.lib.roctxRangePop()


ROCTX = _Roctx()


# ------------------------------------------------------------------ workloads


def run_fit(args, torch):
    from impuritymodel_amd import engine
    from impuritymodel_amd import surrogate as S
    from impuritymodel_amd.batched import plain_xas

    fam = S.XASFamily()
    sur, info = S.train_surrogate(fam, n_train=args.n_train, epochs=args.epochs, seed=0)
    print("set-up: %s" % json.dumps({k: (round(v, 4) if isinstance(v, float) else v) for k, v in info.items()}),
          file=sys.stderr, flush=True)
    target_theta = S.sample_params(1, seed=99)[0]
    target = S.exact_spectra(fam, target_theta[None])[0][0]

    def timed_loop(surrogate, tag, timing):
        # timing: per-kernel HIP events around direct launches (no graphs)
        engine.timing_enable(timing)
        if surrogate is not None:  # walkers stepped inside the library, one call per step
            loop = S.NativeFittingLoop(fam, target, surrogate, n_walkers=args.walkers, seed=1)
        else:
            loop = S.FittingLoop(fam, target, None, n_walkers=args.walkers, seed=1)
        for _ in range(args.warmup):
            loop.step()
        loop.finish()
        torch.cuda.synchronize()
        engine.timing_reset()
        loop.reset_counters()
        torch.cuda.synchronize()
        ROCTX.push(tag)
        t0 = time.perf_counter()
        for _ in range(args.steps):
            loop.step()
        loop.finish()  # proposals still waiting for exact ED are evaluated inside the timed region
        torch.cuda.synchronize()
        dt = time.perf_counter() - t0
        ROCTX.pop()
        kern = {k: engine.timing_query(k) for k in KERNELS}
        engine.timing_enable(False)
        return loop, dt, kern

    # the measured loops run as the product does (kernel timing off, graphs
    # replayed); the same loops again (same seeds, same walk) with per-kernel
    # HIP events give the kernels' average durations for the rooflines
    loop_s, dt_s, _ = timed_loop(sur, "fit_timed_surrogate", False)
    loop_e, dt_e, _ = timed_loop(None, "fit_timed_exact", False)
    loop_si, dt_si, kern_s = timed_loop(sur, "fit_instrumented_surrogate", True)
    loop_ei, dt_ei, kern_e = timed_loop(None, "fit_instrumented_exact", True)
    assert (loop_si.n_spectra, loop_si.n_predicted) == (loop_s.n_spectra, loop_s.n_predicted)
    value = loop_s.n_spectra / dt_s
    batched_rate = loop_e.n_spectra / dt_e
    print("timed: surrogate loop %.3f s (%d spectra, %d by surrogate), exact loop %.3f s; instrumented %.3f s, %.3f s"
          % (dt_s, loop_s.n_spectra, loop_s.n_surrogate, dt_e, dt_si, dt_ei), file=sys.stderr, flush=True)

    # plain GPU ED: one model and one chain at a time, same proposals
    plainP = S.sample_params(args.plain_sample, seed=123)
    t0 = time.perf_counter()
    plain = [S.area_normalize(plain_xas(m, omega=S.OMEGA, delta=S.DELTA, krylovSize=200, T=p[7]))
             for m, p in zip(fam.models(plainP), plainP)]
    plain_rate = len(plainP) / (time.perf_counter() - t0)
    batched_same = S.exact_spectra(fam, plainP)[0]
    plain_vs_batched = float(np.abs(np.array(plain) - batched_same).max())

    # score every surrogate-served spectrum against exact ED
    sp, ss = loop_s.served()
    if len(sp):
        exact = np.concatenate([S.exact_spectra(fam, sp[i:i + 4096])[0] for i in range(0, len(sp), 4096)])
        l1 = S.l1_error(ss, exact)
        score = dict(n=int(len(l1)), l1_max=float(l1.max()), l1_mean=float(l1.mean()),
                     l1_p99=float(np.percentile(l1, 99)), frac_le_1e_2=float((l1 <= 1e-2).mean()))
    else:
        score = dict(n=0)

    # algorithmic bytes of the exact-ED kernels inside the timed surrogate loop
    gs_item = eigen_itemsize(fam)

    def ed_bytes(loop):
        eig = sum(algorithmic_bytes_eigen(r.ground_dims, r.ground_nnz, r.eig_steps) for r in loop.exact_results)
        lan = sum(algorithmic_bytes_lanczos(r.chain_dims, r.chain_nnz, r.kout) for r in loop.exact_results)
        return {"eigen": eig, "lanczos": lan}

    def gs_rate(loop, kern):
        # the eigensolver's Gram-Schmidt reads of Krylov vectors on the chip
        # (registers, then LDS), per second of its launches
        ms, k = kern["eigen"]
        if not k:
            return None
        b = sum(gram_schmidt_bytes(r.ground_dims, r.eig_steps, gs_item) for r in loop.exact_results)
        return dict(kernel=KERNEL_NAMES["eigen"], gram_schmidt_gbs=round(b / (ms * 1e-3) / 1e9, 1),
                    what="classical Gram-Schmidt reads of the stored Krylov vectors (registers, LDS), one pass per step; "
                         "not HBM traffic, not in the roofline")

    # surrogate GEMMs: 2 flops per multiply-add, every layer, every member, every predicted sample
    dims = sur.net.dims
    gemm_flops = 2.0 * sur.net.E * sum(dims[l] * dims[l + 1] for l in range(len(dims) - 1)) * loop_si.n_predicted
    roofline = _roofline(kern_s, ed_bytes(loop_si), {"mlp_gemm": gemm_flops})
    # the exact-ED eigensolver where it dominates: the batched-ED-only loop
    roofline_ed = _roofline({"eigen": kern_e["eigen"]}, ed_bytes(loop_ei))
    if roofline_ed is not None:
        roofline_ed["gram_schmidt"] = gs_rate(loop_ei, kern_e)

    cpu = None
    if not args.no_cpu_baseline:
        workers = args.cpu_workers or min(16, os.cpu_count() or 1)
        cpu = cpu_baseline(_oracle_family, [tuple(p) for p in S.sample_params(5 * workers, seed=321)], workers,
                           "fitting-loop spectra (10-bath family, uniform parameters; the reference's plain "
                           "Lanczos recurrence)")
    peaks = measured_peaks(torch)
    return {
        "metric": METRIC,
        "value": round(value, 3),
        "unit": "spectra/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(1e3 * dt_s / args.steps, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        # surrogate GEMMs in BF16 (FP32 accumulate), statistics and every exact-ED kernel in FP64
        "dtype": "bf16+f64",
        "data": "synthetic (seeded parameters; exact spectra from the engine itself)",
        "config": {
            "workload": "fitting loop: %d Metropolis walkers over 8 parameters of a NiO-like 10-bath model "
                        "(26 spin-orbitals), one XAS per proposal (3 eigenstates, 3 polarizations, Lanczos 200, "
                        "%d omega points, delta %.2f eV, complex128); surrogate = 5 x MLP 8-512-512-512-%d "
                        "(BF16 MFMA, FP32 accumulate), exact fallback by batched ED; walkers stepped in libimped "
                        "(imped_walkers_step: proposals, one prediction with device misfits, decisions)"
                        % (args.walkers, len(S.OMEGA), S.DELTA, len(S.OMEGA)),
            "walkers": args.walkers,
            "spectra_timed": int(loop_s.n_spectra),
            "exact_flushes_timed": int(loop_s.n_flushes),
            "exact_only_spectra_timed": int(loop_e.n_spectra),
            "surrogate_fraction": round(loop_s.n_surrogate / max(loop_s.n_spectra, 1), 4),
            "surrogate_l1_vs_exact": score,
            "batched_ed_only_spectra_per_s": round(batched_rate, 3),
            "plain_gpu_ed_spectra_per_s": round(plain_rate, 4),
            "plain_sample": int(len(plainP)),
            "plain_vs_batched_max_abs_diff": plain_vs_batched,
            "speedup_vs_plain_gpu_ed": round(value / plain_rate, 2),
            "speedup_batched_ed_vs_plain": round(batched_rate / plain_rate, 2),
            "setup": {k: (round(v, 4) if isinstance(v, float) else v) for k, v in info.items()},
            "kernel_timing": "per-kernel HIP events in an identical repeat of each timed loop (same seeds and "
                             "walk, direct launches); the timed loops themselves run uninstrumented",
            "instrumented_loop_seconds": {"surrogate": round(dt_si, 4), "exact_only": round(dt_ei, 4)},
            "kernel_ms_per_step": {k: round(v[0] / args.steps, 4) for k, v in kern_s.items() if v[1]},
            "kernel_ms_per_step_exact_loop": {k: round(v[0] / args.steps, 4) for k, v in kern_e.items() if v[1]},
            "roofline_eigen_exact_loop": roofline_ed,
            "measured_peaks": peaks,
        },
        "roofline": roofline,
        "cpu_baseline": cpu,
    }


def run_exact(args, torch):
    """The fitting family's exact path alone: ``--models`` proposals per batched
    exact-ED call (the call that answers the surrogate's untrusted proposals),
    no surrogate and no training."""
    from impuritymodel_amd import engine
    from impuritymodel_amd import surrogate as S

    fam = S.XASFamily()
    P = [S.sample_params(args.models, seed=1000 + k) for k in range(args.steps + args.warmup)]
    for k in range(args.warmup):
        S.exact_spectra(fam, P[k], sectors=not args.general_path)
    torch.cuda.synchronize()
    ROCTX.push("exact_timed")
    t0 = time.perf_counter()
    for k in range(args.steps):
        S.exact_spectra(fam, P[args.warmup + k], sectors=not args.general_path)
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    ROCTX.pop()
    engine.timing_enable(True)
    engine.timing_reset()
    ROCTX.push("exact_instrumented")
    results = [S.exact_spectra(fam, P[args.warmup + k], sectors=not args.general_path)[1] for k in range(args.steps)]
    torch.cuda.synchronize()
    ROCTX.pop()
    kernels = {k: engine.timing_query(k) for k in KERNELS + ("discover", "sort", "csr_fill", "affine_fill",
                                                              "affine_seed")}
    engine.timing_enable(False)
    # the same proposals through the other path (the general path, or with
    # --general-path the sector cache)
    nb = min(args.steps, 5)
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    for k in range(nb):
        S.exact_spectra(fam, P[args.warmup + k], sectors=args.general_path)
    torch.cuda.synchronize()
    other_ms = 1e3 * (time.perf_counter() - t1) / nb
    eig = sum(algorithmic_bytes_eigen(r.ground_dims, r.ground_nnz, r.eig_steps) for r in results)
    lan = sum(algorithmic_bytes_lanczos(r.chain_dims, r.chain_nnz, r.kout) for r in results)
    # the per-step byte models describe the Krylov kernels; a chain solved
    # by a Householder reduction (eigen_dense_max_n, lanczos_dense_max_n)
    # has no such model, so its kernel is left out of the roofline
    tuned = dict((kv.split("=", 1)[0], int(kv.split("=", 1)[1])) for kv in args.tuning)
    krylov = [k for k, knob in (("eigen", "eigen_dense_max_n"), ("lanczos", "lanczos_dense_max_n"))
              if tuned.get(knob, 0) <= 0]
    roofline = _roofline({k: kernels[k] for k in krylov}, {"eigen": eig, "lanczos": lan},
                         workload="exact%d" % args.models) if krylov else None
    if roofline is not None and roofline["kernel"] == KERNEL_NAMES["eigen"]:
        b = sum(gram_schmidt_bytes(r.ground_dims, r.eig_steps, eigen_itemsize(fam)) for r in results)
        roofline["gram_schmidt_gbs"] = round(b / (kernels["eigen"][0] * 1e-3) / 1e9, 1)
    r0 = results[-1]
    return {
        "metric": METRIC,
        "value": round(args.models * args.steps / dt, 3),
        "unit": "spectra/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(1e3 * dt / args.steps, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (seeded parameters)",
        "config": {
            "workload": "exact path of the fitting loop: %d proposals of the NiO-like 10-bath family per batched "
                        "exact-ED call (3 eigenstates, 3 polarizations, fully reorthogonalized Lanczos, 1000 "
                        "omega points), no surrogate" % args.models,
            "models_per_call": args.models,
            "path": "general (every sector rebuilt per call)" if args.general_path else
                    "family sector cache (patterns fixed, values and start vectors formed per call)",
            "ground_chains_per_model": len(r0.ground_dims) // args.models,
            "ground_dims": sorted(set(int(x) for x in r0.ground_dims)),
            "ground_nnz": sorted(set(int(x) for x in r0.ground_nnz)),
            "excited_dims": sorted(set(int(x) for x in r0.chain_dims)),
            ("sector_cache_ms_per_call" if args.general_path else "general_path_ms_per_call"): round(other_ms, 3),
            "chains_per_call": int(len(r0.chain_dims)),
            "eigen_steps_range": [int(min(r.eig_steps.min() for r in results)),
                                  int(max(r.eig_steps.max() for r in results))],
            "kernel_timing": "HIP events around every launch in a repeat of the timed calls",
            "kernel_ms_per_call": {k: round(v[0] / args.steps, 4) for k, v in kernels.items() if v[1]},
            "launches_per_call": {k: v[1] // args.steps for k, v in kernels.items() if v[1]},
        },
        "roofline": roofline,
        "cpu_baseline": None,
    }


def run_large(args, torch):
    """Large single instance: 76 spin-orbitals (two words per state), sectors of ~10^6 states."""
    from impuritymodel_amd import engine
    from impuritymodel_amd.batched import POLARIZATIONS, ground_bases, state_spectra
    from impuritymodel_amd.engine import Batch, Ops
    from impuritymodel_amd.models import K_B, large_model
    from impuritymodel_amd.operators import getDipoleOperators, getNIXSOperators, getPhotoEmissionOperators

    m = large_model()
    n, W = m.n_spin_orbitals, 2
    ops_h = Ops([m.hOp], [m.restrictions], n, W)
    ops_xas = Ops(getDipoleOperators(m.nBaths, POLARIZATIONS), [m.restrictions] * 3, n, W)
    omega = np.linspace(-25.0, 25.0, 3000)
    K = 300

    def ground():
        basis = ground_bases([m], W)[0]
        gb = Batch(ops_h, [0])
        gb.set_seeds([basis])
        t0 = time.perf_counter()
        gb.build(fixed_basis=True)
        torch.cuda.synchronize()
        t_build = time.perf_counter() - t0
        t0 = time.perf_counter()
        ev, _, steps, _ = gb.eigen(3, tol=1e-12, max_steps=600, want_vectors=False)
        torch.cuda.synchronize()
        t_eig = time.perf_counter() - t0
        e = ev[0]
        kept = [i for i in range(3) if e[i] - e[0] < 10.0 * K_B * 300.0]
        psis = gb.vec_from_eigen(np.zeros(len(kept), np.int32), np.array(kept, np.int32), 1e-7)
        return gb, e[kept], psis, t_build, t_eig, int(steps[0])

    def xas_step(label):
        t0 = time.perf_counter()
        gb, es, psis, t_build, t_eig, steps = ground()
        print("large %s: ground state done (%.2f s)" % (label, time.perf_counter() - t0), file=sys.stderr, flush=True)
        spec, info = state_spectra(ops_h, ops_xas, psis, es, omega, 0.2, K, T=300.0)
        torch.cuda.synchronize()
        print("large %s: XAS done (%.2f s)" % (label, time.perf_counter() - t0), file=sys.stderr, flush=True)
        return time.perf_counter() - t0, gb, es, psis, t_build, t_eig, steps, spec, info

    for _ in range(args.warmup):
        xas_step("warm-up")
    # timed steps: launch timing off, so the Lanczos steps replay as HIP graphs
    torch.cuda.synchronize()
    ROCTX.push("large_timed")
    t0 = time.perf_counter()
    runs = [xas_step("timed") for _ in range(args.steps)]
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    ROCTX.pop()
    _, gb, es, psis, t_build, t_eig, eig_steps, spec, info = runs[-1]
    # one more step with launch timing on (every launch direct, each timed by
    # HIP events on the engine's stream): per-kernel durations for the roofline
    engine.timing_enable(True)
    engine.timing_reset()
    ROCTX.push("large_instrumented")
    _, gb_i, _, _, _, _, eig_steps_i, _, info_i = xas_step("instrumented")
    ROCTX.pop()
    kernels = {k: engine.timing_query(k)
               for k in ("spmv", "eigen_flat", "apply_count", "apply_fill", "discover", "sort", "csr_fill", "cf")}
    engine.timing_enable(False)
    # Hamiltonian builds of the instrumented step (ground fixed-basis build and
    # the BFS closures of the XAS sectors): 8 W n + 20 nnz + 4 (n + 1) bytes
    # each (basis keys read, CSR written), over the build kernels' time
    build_kernels = ("apply_count", "apply_fill", "discover", "sort", "csr_fill")
    build_ms = sum(kernels[k][0] for k in build_kernels)
    bb = lambda nn, zz: 8.0 * W * nn + 20.0 * zz + 4.0 * (nn + 1)
    build_bytes = bb(gb_i.rows, gb_i.nnz) + sum(bb(nn, zz) for nn, zz in zip(info_i["chain_n"], info_i["chain_nnz"]))
    build = dict(kernels=list(build_kernels), kernel_ms=round(build_ms, 3), algorithmic_bytes=build_bytes,
                 achieved_gbs=round(build_bytes / (build_ms * 1e-3) / 1e9, 1) if build_ms else None,
                 frac=round(build_bytes / (build_ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4) if build_ms else None,
                 states=int(gb_i.rows + int(np.sum(info_i["chain_n"]))),
                 states_per_s=round((gb_i.rows + float(np.sum(info_i["chain_n"]))) / (build_ms * 1e-3), 1)
                 if build_ms else None)
    # algorithmic bytes of every flat SpMV launch in the instrumented step: the
    # Lanczos chains (K steps each, complex vectors) and the ground-state
    # eigensolver (eig_steps SpMVs, real vectors when H is real); per launch
    # (value + 4) nnz + 8 (n+1) + 2 n (vector element) bytes: int32 columns,
    # int64 row pointers, x read once, y written.  A real H is read as 8-byte
    # values (the real_values knob, on by default), else as complex128.
    h_real = not any(complex(v).imag for v in m.hOp.values())
    vb = 8.0 if h_real and _tuning_value(args, "real_values", 1) else 16.0
    eb = 8.0 if h_real and _tuning_value(args, "eigen_real", 1) else 16.0
    spmv_bytes = lambda nn, zz, xb: (vb + 4.0) * zz + 8.0 * (nn + 1) + 2.0 * xb * nn
    per_step = sum(int(k) * spmv_bytes(nn, zz, 16.0)
                   for nn, zz, k in zip(info_i["chain_n"], info_i["chain_nnz"], info_i["kout"]))
    per_step += eig_steps_i * spmv_bytes(gb_i.rows, gb_i.nnz, eb)
    roofline = _roofline({"spmv": kernels["spmv"]}, {"spmv": per_step},
                         workload="large_real" if vb == 8.0 else "large_complex")
    roofline["measured_on"] = "one instrumented step after the timed ones (launch timing forces direct launches)"

    # XPS (2p removal, photoemission convention) and NIXS (|q| = 2, 7 along (111), 3d -> 3d: k = 2, 4)
    extra = {}
    if args.no_extras:
        return _large_result(args, dt, gb, t_build, t_eig, eig_steps, info, kernels, extra, roofline, build)
    ops_xps = Ops(getPhotoEmissionOperators(m.nBaths, l=1), [m.restrictions] * 6, n, W)
    t0 = time.perf_counter()
    _, xinfo = state_spectra(ops_h, ops_xps, psis, es, omega, 0.2, K, T=300.0, sign=-1)
    torch.cuda.synchronize()
    extra["xps"] = dict(seconds=round(time.perf_counter() - t0, 4), chains=int(len(xinfo["chain_n"])),
                        chain_n_max=int(xinfo["chain_n"].max()))
    r, R = np.loadtxt(os.path.join(ROOT, "tests", "golden", "Ni3d.dat")).T
    qs = [2.0 * np.ones(3) / np.sqrt(3.0), 7.0 * np.ones(3) / np.sqrt(3.0)]
    ops_nixs = Ops(getNIXSOperators(m.nBaths, qs, 2, 2, R, R, r), [m.restrictions] * 2, n, W)
    t0 = time.perf_counter()
    _, ninfo = state_spectra(ops_h, ops_nixs, psis, es, omega, 0.2, K, T=300.0)
    torch.cuda.synchronize()
    extra["nixs"] = dict(seconds=round(time.perf_counter() - t0, 4), chains=int(len(ninfo["chain_n"])),
                         chain_n_max=int(ninfo["chain_n"].max()), q_norms=[2.0, 7.0], l_i=2, l_j=2, k=[2, 4])
    return _large_result(args, dt, gb, t_build, t_eig, eig_steps, info, kernels, extra, roofline, build)


def _large_result(args, dt, gb, t_build, t_eig, eig_steps, info, kernels, extra, roofline, build):
    return {
        "metric": METRIC,
        "value": round(args.steps / dt, 4),
        "unit": "spectra/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(1e3 * dt / args.steps, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (seeded parameters)",
        "config": {
            "workload": "large single instance: NiO-like model with 50 valence + 10 conduction bath spin-orbitals "
                        "(76 spin-orbitals, 2 words per state); per step: ground basis, fixed-basis H, 3 lowest "
                        "eigenstates (tol 1e-12), 3 dipole polarizations x kept states, BFS closure + CSR of "
                        "every XAS sector, 300-step Lanczos, continued fractions on 3000 omega points; complex128",
            "ground_states": int(gb.rows), "ground_nnz": int(gb.nnz),
            "ground_build_s": round(t_build, 4),
            "ground_build_states_per_s": round(gb.rows / t_build, 1),
            "ground_eigen_s": round(t_eig, 4), "ground_eigen_steps": eig_steps,
            "xas_chains": int(len(info["chain_n"])), "xas_chain_n": [int(x) for x in info["chain_n"]],
            "xas_chain_nnz": [int(x) for x in info["chain_nnz"]],
            "xas_build_s": round(info["build_s"], 4),
            "xas_build_states_per_s": round(float(info["chain_n"].sum()) / info["build_s"], 1),
            "xas_lanczos_s": round(info["lanczos_s"], 4), "xas_cf_s": round(info["cf_s"], 4),
            "kernel_ms_instrumented_step": {k: round(v[0], 3) for k, v in kernels.items() if v[1]},
            "build_kernels_hbm": build,
            "extra_spectra": extra,
        },
        "roofline": roofline,
        "cpu_baseline": None,
    }


def run_rixs(args, torch):
    """Batched RIXS map of a 20-bath model against the per-incoming-energy path."""
    from impuritymodel_amd import engine
    from impuritymodel_amd.batched import POLARIZATIONS, ground_bases
    from impuritymodel_amd.engine import Batch, Ops
    from impuritymodel_amd.models import K_B, make_model
    from impuritymodel_amd.operators import getDaggeredDipoleOperators, getDipoleOperators
    from impuritymodel_amd.spectra import _rixs_chains

    m = make_model(n_bath=20, seed=11)
    n = m.n_spin_orbitals
    W = 1
    ops_h = Ops([m.hOp], [m.restrictions], n, W)
    tin = Ops(getDipoleOperators(m.nBaths, POLARIZATIONS), [m.restrictions] * 3, n, W)
    tout = Ops(getDaggeredDipoleOperators(m.nBaths, POLARIZATIONS), [m.restrictions] * 3, n, W)
    w_in = np.linspace(-5.0, 15.0, 64)
    w_loss = np.linspace(-2.0, 13.0, 1500)
    gamma, delta2, K = 0.5, 0.1, 150
    # out-going chains fully reorthogonalized: the plain recurrence past loss of
    # orthogonality turns the 1e-12 differences of the two solve paths into
    # 1e-6 differences of the map
    REORTH = "full"

    def rixs_map(plain=False):
        gb = Batch(ops_h, [0])
        gb.set_seeds(ground_bases([m], W))
        gb.build(fixed_basis=True)
        ev, _, _, _ = gb.eigen(3, tol=1e-12, max_steps=600, want_vectors=False)
        e = ev[0]
        kept = [i for i in range(3) if e[i] - e[0] < 10.0 * K_B * 300.0]
        psis = gb.vec_from_eigen(np.zeros(len(kept), np.int32), np.array(kept, np.int32), 1e-7)
        es = e[kept]
        if not plain:
            g, tim = _rixs_chains(n, ops_h, tin, tout, psis, es, 3, 3, w_in, w_loss, gamma, delta2, K, 1e-7, False,
                                  REORTH, 1e-12, 1000)
        else:
            parts = []
            tim = {}
            for w in w_in:
                gi, _ = _rixs_chains(n, ops_h, tin, tout, psis, es, 3, 3, np.array([w]), w_loss, gamma, delta2, K,
                                     1e-7, False, REORTH, 1e-12, 1000)
                parts.append(gi)
            g = np.concatenate(parts, axis=3)
        # thermal average over eigenstates, summed over polarization pairs
        wts = np.exp(-(es - es.min()) / (K_B * 300.0))
        amap = np.einsum("e,eabwl->wl", wts / wts.sum(), -g.imag)
        return amap, tim, len(kept)

    for _ in range(args.warmup):
        rixs_map()
    engine.timing_enable(True)
    engine.timing_reset()
    torch.cuda.synchronize()
    ROCTX.push("rixs_timed")
    t0 = time.perf_counter()
    maps = [rixs_map() for _ in range(args.steps)]
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    ROCTX.pop()
    kernels = {k: engine.timing_query(k) for k in ("solve", "solve_combine", "lanczos", "eigen", "apply_count",
                                                   "apply_fill", "cf")}
    engine.timing_enable(False)
    amap, tim, n_kept = maps[-1]
    t0 = time.perf_counter()
    pmap, _, _ = rixs_map(plain=True)
    t_plain = time.perf_counter() - t0
    rel = float(np.abs(amap - pmap).max() / np.abs(pmap).max())
    return {
        "metric": METRIC,
        "value": round(args.steps / dt, 4),
        "unit": "RIXS maps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(1e3 * dt / args.steps, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (seeded parameters)",
        "config": {
            "workload": "batched RIXS map: NiO-like 20-bath model (46 spin-orbitals), 64 incoming energies in "
                        "[-5, 15] eV (Gamma 0.5 eV) solved from one Krylov space per (T_in, eigenstate), 3 x 3 "
                        "polarization pairs, out-going 150-step Lanczos, 1500 loss points (delta 0.1 eV); "
                        "complex128",
            "eigenstates": n_kept,
            "out_going_chains": int(n_kept * 9 * len(w_in)),
            "stage_s": {k: round(float(v), 4) for k, v in tim.items() if np.ndim(v) == 0},
            "chain_n_range": {k: [int(np.min(v)), int(np.max(v))] for k, v in tim.items() if np.ndim(v) > 0 and len(v)},
            "plain_per_energy_s": round(t_plain, 3),
            "speedup_vs_plain": round(t_plain / (dt / args.steps), 2),
            "map_rel_diff_vs_plain": rel,
            "kernel_ms_per_step": {k: round(v[0] / args.steps, 3) for k, v in kernels.items() if v[1]},
        },
        "roofline": None,
        "cpu_baseline": None,
    }


def run_batched128(args, torch):
    from impuritymodel_amd import engine
    from impuritymodel_amd.batched import ground_bases, plain_xas, xas_batch
    from impuritymodel_amd.engine import Batch, Ops
    from impuritymodel_amd.models import batched_params, model_from_params

    params = batched_params(args.models, seed=0)
    models = [model_from_params(p) for p in params]
    omega = np.linspace(-25.0, 25.0, 2000)
    n_orb = max(m.n_spin_orbitals for m in models)
    gb_ops = Ops([m.hOp for m in models], [m.restrictions for m in models], n_orb)
    gb = Batch(gb_ops, np.arange(len(models), dtype=np.int32))
    gb.set_seeds(ground_bases(models, gb_ops.W))
    gb.build(fixed_basis=True)
    tuned = None
    if not args.no_autotune:
        # untimed: the eigensolver's launch shapes (threads per chain, Ritz
        # check interval, one-wave bucket) timed on this workload's own ground
        # chains; the timed steps run with the fastest of each
        from impuritymodel_amd import autotune

        t_tune = time.perf_counter()
        table = autotune.autotune(eigen_batch=gb, nev=3, repeats=2)
        tuned = {"seconds": round(time.perf_counter() - t_tune, 3), "table": table}
    for _ in range(args.warmup):
        res = xas_batch(models, omega=omega, krylovSize=200)
    torch.cuda.synchronize()
    # timed steps as the product runs them (no kernel timing)
    ROCTX.push("batched128_timed")
    t0 = time.perf_counter()
    for _ in range(args.steps):
        res = xas_batch(models, omega=omega, krylovSize=200)
    torch.cuda.synchronize()
    dt = time.perf_counter() - t0
    ROCTX.pop()
    # the same steps again with a HIP-event pair around every launch
    engine.timing_enable(True)
    engine.timing_reset()
    ROCTX.push("batched128_instrumented")
    for _ in range(args.steps):
        res = xas_batch(models, omega=omega, krylovSize=200)
    torch.cuda.synchronize()
    ROCTX.pop()
    kernels = {k: engine.timing_query(k) for k in KERNELS}
    engine.timing_enable(False)
    roofline = _roofline(kernels, {
        "eigen": args.steps * algorithmic_bytes_eigen(gb.chain_n, gb.chain_nnz, res.eig_steps),
        "lanczos": args.steps * algorithmic_bytes_lanczos(res.chain_dims, res.chain_nnz, res.kout)},
        # mixed sizes: a class's launches are those of two kernels
        names={"eigen": "eigen_reg_kernel + eigen_kernel", "lanczos": "lanczos_reg_kernel + lanczos_kernel"})
    # plain GPU ED (one model, one chain per launch sequence) on a sample of the same models
    idx = list(range(0, args.models, max(1, args.models // args.plain_sample)))[: args.plain_sample]
    t0 = time.perf_counter()
    plain = [plain_xas(models[i], omega=omega, krylovSize=200) for i in idx]
    torch.cuda.synchronize()
    plain_rate = len(idx) / (time.perf_counter() - t0)
    plain_diff = max(float(np.abs(p - res.spectra[i]).max() / np.abs(res.spectra[i]).max()) for p, i in zip(plain, idx))
    value = args.models * args.steps / dt
    cpu = None
    if not args.no_cpu_baseline:
        workers = args.cpu_workers or min(16, os.cpu_count() or 1)
        items = [(params[i % len(params)], omega, 200) for i in range(2 * workers)]
        cpu = cpu_baseline(_oracle_batched, items, workers, "models of the same parameter distribution", per_worker=1)
    return {
        "metric": METRIC,
        "value": round(value, 3),
        "unit": "spectra/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(1e3 * dt / args.steps, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic (seeded impurity-model parameters)",
        "config": {
            "workload": "batched exact-diagonalization XAS, %d NiO-like impurity models per step (bath sizes "
                        "10-50 spin-orbitals, 26-66 spin-orbitals), 3 polarizations x <=3 thermal states, "
                        "Lanczos 200 steps (fully reorthogonalized), 2000 omega points, complex128; exact path "
                        "(no surrogate)" % args.models,
            "models_per_step": args.models,
            "chains_per_step": int(len(res.chain_dims)),
            "chain_dim_range": [int(res.chain_dims.min()), int(res.chain_dims.max())],
            "plain_gpu_ed_spectra_per_s": round(plain_rate, 3),
            "plain_sample": len(idx),
            "speedup_batched_vs_plain_gpu_ed": round(value / plain_rate, 2),
            "plain_vs_batched_max_rel_diff": plain_diff,
            "kernel_timing": "HIP events around every launch in a repeat of the timed steps",
            "kernel_ms_per_step": {k: round(v[0] / args.steps, 3) for k, v in kernels.items() if v[1]},
            "autotune": tuned if tuned is not None else "off (--no-autotune): default launch shapes",
        },
        "roofline": roofline,
        "cpu_baseline": cpu,
    }


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20, help="timed steps")
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--workload", choices=("fit", "exact", "batched128", "large", "rixs"), default="fit")
    ap.add_argument("--models", type=int, default=128)
    ap.add_argument("--general-path", action="store_true",
                    help="exact workload: rebuild every sector per call instead of the family sector cache")
    ap.add_argument("--walkers", type=int, default=256)
    ap.add_argument("--n-train", type=int, default=20000)
    ap.add_argument("--epochs", type=int, default=2500)
    ap.add_argument("--plain-sample", type=int, default=8)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-autotune", action="store_true",
                    help="batched128: time with the default launch shapes instead of the autotuned ones")
    ap.add_argument("--cpu-workers", type=int, default=0)
    ap.add_argument("--no-extras", action="store_true", help="large workload: skip the XPS/NIXS extras")
    ap.add_argument("--calibration-copy-mib", type=int, default=0,
                    help="copy this many MiB device-to-device first (counter calibration under rocprofv3 --pmc)")
    ap.add_argument("--tuning", action="append", default=[], metavar="NAME=VALUE",
                    help="set an engine launch-shape knob (imped_set_tuning) before the run; repeatable")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU only: the engine runs on a single MI355X; "
              "--gpus %d is not supported" % args.gpus, file=sys.stderr)
        sys.exit(2)

    import torch

    assert torch.cuda.is_available(), "bench.py needs a GPU"
    torch.cuda.set_device(0)
    if args.calibration_copy_mib:
        # one device copy of known size: the scale of the FETCH_SIZE/WRITE_SIZE
        # counters against true bytes when the run is profiled with --pmc
        nbytes = args.calibration_copy_mib << 20
        src = torch.ones(nbytes // 4, dtype=torch.float32, device="cuda")
        dst = torch.empty_like(src)
        dst.copy_(src)
        # the same bytes through a plain streaming elementwise kernel
        torch.mul(src, 1.0, out=dst)
        torch.cuda.synchronize()
        del src, dst
    if args.tuning:
        from impuritymodel_amd import engine

        for kv in args.tuning:
            name, value = kv.split("=", 1)
            engine.set_tuning(name, int(value))
    run = {"fit": run_fit, "exact": run_exact, "batched128": run_batched128, "large": run_large,
           "rixs": run_rixs}[args.workload]
    out = run(args, torch)
    if args.tuning:
        out["config"]["tuning"] = dict(kv.split("=", 1) for kv in args.tuning)
    print(json.dumps(out))


if __name__ == "__main__":
    main()
