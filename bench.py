"""Benchmark: seconds to all eigenpairs of an n = 32768 FP64 symmetric tridiagonal
(d, e ~ U(-1,1), seed 2; HSS leaf 128, tolerance 1e-13, HSS branch for K >= 1024)
with the batched divide-and-conquer path and the learned secular start on one
MI355X, device resident.

One step = one complete solve (eigenvalues and the n x n eigenvector matrix) with
the input already in HBM; `value` times the solve as used (levels queued at once,
replayed as a HIP graph).  Prints one JSON line.  Also in the line:
  * a profiled pass of the same solve (direct launches, HIP events) giving the
    roofline of the dominant kernel -- the zero fill of the output, on a second stream
    beside the DC levels -- and the rates of the hot-path kernels (secular sweep and
    Loewner / alpha sweeps in GB/s of their algorithmic bytes, the HSS multiply in
    TFLOP/s, the HSS construction against HSSPACK's flop model);
  * ablations: classical secular start, a host round trip per level, the
    merge-at-a-time ("plain") schedule; orthogonality and residual; the host-to-host
    time of the host-array entry (Z copied back);
  * config.hss_workload: the same for the n = 32768 near-Toeplitz matrix (63 HSS merges,
    learned start active) at HSS tolerance 1e-15 and 1e-13;
  * CPU baselines on the host's threads: the oracle (restatement of the reference path)
    and LAPACK dstedc.

usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--cfg 1 --seed 4]
                       [--no-cpu] [--no-plain] [--no-check] [--no-hss]
                       [--batch | --svd [--svd-toeplitz] | --band [--kd 64]]
"""
import argparse
import ctypes
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
FP64_PEAK_TFS = 78.6
# HBM bytes per k_zfill launch measured with rocprofv3 FETCH_SIZE / WRITE_SIZE passes, calibrated on a
# 1 GiB device copy (profiles/k_zfill_n32768_uniform_traffic.md); keyed by (generator, n, seed)
K_ZFILL_TRAFFIC = {(2, 32768, 2): (40 + 8388627) * 1024}
GEN = {1: "d=2+U(-1e-3,1e-3), e=1+U(-1e-3,1e-3)", 2: "d,e~U(-1,1)"}


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def check_result(torch, d, e, lam, zz):
    """max|Z'Z - I| and max|TZ - Z diag(lam)| / max|T| on the device.
    zz holds Z column-major, i.e. zz[j, :] is eigenvector j."""
    n = zz.shape[0]
    dev = zz.device
    dd = torch.tensor(d, device=dev)
    ee = torch.tensor(e, device=dev)
    orth = 0.0
    blk = 4096
    for i0 in range(0, n, blk):
        g = zz[i0:i0 + blk] @ zz.T
        g[:, i0:i0 + blk].diagonal().sub_(1.0)
        orth = max(orth, g.abs().max().item())
        del g
    lam_t = torch.tensor(lam, device=dev)
    res = 0.0
    for i0 in range(0, n, blk):
        z = zz[i0:i0 + blk]
        tz = z * dd
        tz[:, 1:] += z[:, :-1] * ee
        tz[:, :-1] += z[:, 1:] * ee
        tz -= z * lam_t[i0:i0 + blk, None]
        res = max(res, tz.abs().max().item())
    nrm = max(abs(d).max(), abs(e).max())
    return float(orth), float(res / nrm)


MLP_FILE = os.path.join(ROOT, "hsspack_amd", "data", "secular_mlp.bin")


def host_threads():
    """Threads the CPU baselines use: OMP_NUM_THREADS when set (16 on the GPU host), else every core."""
    return int(os.environ.get("OMP_NUM_THREADS") or os.cpu_count() or 1)


def cpu_model():
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def _extrapolate(np, times, n_full):
    (n0, t0), (n1, t1) = sorted(times.items())
    p = np.log(t1 / t0) / np.log(n1 / n0)
    return t1 * (n_full / float(n1)) ** p, p


def cpu_baseline(cfg, seed, hss, n_full):
    """The oracle (C restatement of the reference path) on the same generator, with OpenMP
    over the loops whose outputs are independent (GEMM columns, the identity fill, the
    final permutation; the reference runs its GEMMs in threaded BLAS) on host_threads()
    threads.  The headline generator (nearly everything deflates) runs at its full order;
    the HSS-heavy one is timed at 4096 and 8192 and extrapolated with the measured
    exponent (its full order would take about ten minutes)."""
    import numpy as np
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import oracle_py as O
    from hsspack_amd.workloads import tridiag_cfg
    L = O.lib()

    def run(n):
        d, e = tridiag_cfg(cfg, n, seed)
        z = np.zeros((n, n), order="F")
        lwork, liwork = 1 + 4 * n + n * n, 3 + 5 * n
        work = np.zeros(lwork)
        iwork = np.zeros(liwork, np.int32)
        prm = O.params(bsmlz=hss[0], ni=hss[1], tol=hss[2])
        t0 = time.perf_counter()
        info = L.orc_stedc(ctypes.c_char(b"I"), n, O.dp(d), O.dp(e), O.dp(z), n, O.dp(work), lwork,
                           O.ip(iwork), liwork, ctypes.byref(prm), None)
        t = time.perf_counter() - t0
        assert info == 0
        log("cpu oracle n=%d: %.2f s (%d threads)" % (n, t, host_threads()))
        return t

    base = dict(unit="s", cores=host_threads(), cpu=cpu_model(), kind="port")
    what = "oracle (C restatement of mdstedc/mdlaed0-3 + DHSSEVC, OpenMP over independent GEMM columns and copies)"
    if cfg == 2:
        return dict(base, value=run(n_full),
                    sample="%s, the full workload: n=%d, same generator and seed, all eigenpairs" % (what, n_full))
    times = {n: run(n) for n in (4096, 8192)}
    est, p = _extrapolate(np, times, n_full)
    return dict(base, value=est, sample="%s on the same generator at n=4096 (%.2f s) and n=8192 (%.2f s), "
                                        "extrapolated to n=%d with the measured exponent %.2f"
                                        % (what, times[4096], times[8192], n_full, p))


def cpu_lapack(cfg, seed, n_full):
    """LAPACK dstedc (scipy's OpenBLAS, threaded) on the same matrix, all eigenpairs; as
    cpu_baseline, at the full order for the headline generator, extrapolated from 4096
    and 8192 for the HSS-heavy one."""
    import numpy as np
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import lapack_ref as LR
    from hsspack_amd.workloads import tridiag_cfg

    def run(n):
        d, e = tridiag_cfg(cfg, n, seed)
        t0 = time.perf_counter()
        _, z, info = LR.dstedc(d, e)
        t = time.perf_counter() - t0
        assert info == 0
        del z
        log("cpu LAPACK dstedc n=%d: %.2f s" % (n, t))
        return t

    base = dict(unit="s", cores=host_threads(), cpu=cpu_model(), kind="lapack")
    if cfg == 2:
        return dict(base, value=run(n_full), sample="LAPACK dstedc (OpenBLAS 0.3.28), full workload n=%d" % n_full)
    times = {n: run(n) for n in (4096, 8192)}
    est, p = _extrapolate(np, times, n_full)
    return dict(base, value=est, sample="LAPACK dstedc (OpenBLAS 0.3.28) at n=4096 (%.2f s) and 8192 (%.2f s), "
                                        "extrapolated to n=%d with exponent %.2f" % (times[4096], times[8192],
                                                                                     n_full, p))


def secstats(st):
    return {"iters_per_root": st["secular_iters"] / max(st["roots"], 1),
            "wave_iters": st["secular_wave_iters"], "critical_path_iters": st["secular_crit_iters"],
            "learned_roots": st["learned_roots"]}


def bench_tridiag(args, np, torch, hsdc, cfg, n, seed, tol, d, e, steps, warmup, plain=True, check=True,
                  sync_ablation=False, h2h=True):
    """One tridiagonal workload.  value_s: seconds per device-resident solve, the batched
    schedule with the learned start, levels queued at once and replayed as a HIP graph.
    Then a profiled pass of the same solve (direct launches, HIP events around the zero fill,
    the final reordering, the secular, Loewner / alpha and HSS launches) gives the rates,
    and ablations time the classical start, the per-level host round trip and the
    merge-at-a-time schedule."""
    dev = torch.device("cuda:0")
    D0 = torch.tensor(d, device=dev)
    E0 = torch.tensor(np.append(e, 0.0), device=dev)
    D = torch.empty_like(D0)
    E = torch.empty_like(E0)
    Z = torch.empty((n, n), dtype=torch.float64, device=dev)
    ctx = hsdc.Context(hss_min_k=1024, hss_leaf=128, hss_tol=tol, batched=1, learned=1, graph=1, profile=0)
    ctx.mlp_load(MLP_FILE)

    def step():
        D.copy_(D0)
        E.copy_(E0)
        rc = ctx.stedc_dev(D, E, Z)
        if rc != 0:
            raise RuntimeError("hsdc_stedc_dev returned %d" % rc)

    def timed(k):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(k):
            step()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) / k

    for _ in range(warmup):
        step()
    value = timed(steps)
    st = ctx.stats()
    tr = ctx.trace()
    sec_learned = secstats(st)
    log("n=%d tol %g: %.2f ms/solve (graph), stats %s" % (n, tol, value * 1e3, st))
    # profiled pass
    ctx.set_params(profile=1)
    step()
    keys = ("ms_zfill", "ms_final", "ms_secular", "ms_loewner", "ms_hss_build", "ms_hss_mm", "ms_total")
    acc = {k: 0.0 for k in keys}
    nprof = max(2, min(steps, 5))
    t_prof = 0.0
    for _ in range(nprof):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        step()
        torch.cuda.synchronize()
        t_prof += time.perf_counter() - t0
        sp = ctx.stats()
        for k in keys:
            acc[k] += sp[k] / nprof
    ctx.set_params(profile=0)
    t_prof /= nprof
    log("profiled pass: %.2f ms/solve, %s" % (t_prof * 1e3, {k: round(v, 3) for k, v in acc.items()}))

    def rate(nbytes, ms):
        return nbytes / (ms * 1e-3) / 1e9 if ms > 0 else None

    hot = {}
    if sp["secular_evals"] and acc["ms_secular"] > 0:
        b = 16 * sp["secular_evals"]
        hot["k_secular"] = {"bytes": b, "ms": acc["ms_secular"], "GBps": rate(b, acc["ms_secular"]),
                            "frac_of_hbm": rate(b, acc["ms_secular"]) / HBM_PEAK_GBS,
                            "pole_evaluations": sp["secular_evals"],
                            "unit_note": "16 B per pole evaluation (one pole, one z), K evaluations per iteration; "
                                         "with the k_secstart learned-start launches"}
    if sp["loewner_pairs"] and acc["ms_loewner"] > 0:
        b = 16 * sp["loewner_pairs"]
        hot["k_loewner+k_alpha"] = {"bytes": b, "ms": acc["ms_loewner"], "GBps": rate(b, acc["ms_loewner"]),
                                    "frac_of_hbm": rate(b, acc["ms_loewner"]) / HBM_PEAK_GBS,
                                    "pairs": sp["loewner_pairs"],
                                    "unit_note": "16 B per (i, j) operand pair, K^2 per merge for the products, "
                                                 "K^2 more per HSS merge for alpha; the operands are staged in LDS, "
                                                 "so this is an operand rate in HBM units, not HBM traffic: the "
                                                 "sweeps are bound by the FP64 divides"}
    if sp["hss_mm_flops"] and acc["ms_hss_mm"] > 0:
        tf = sp["hss_mm_flops"] / (acc["ms_hss_mm"] * 1e-3) / 1e12
        hot["k_bgemm"] = {"flops": sp["hss_mm_flops"], "ms": acc["ms_hss_mm"], "TFLOPs": tf,
                          "frac_of_fp64_peak": tf / FP64_PEAK_TFS,
                          "unit_note": "2 L (|H| + |DD|) per merge: the DGEMMs of fastHssmmL"}
    if sp["hss_nflops"] and acc["ms_hss_build"] > 0:
        gf = sp["hss_nflops"] / (acc["ms_hss_build"] * 1e-3) / 1e9
        hot["hss_construction"] = {"nflops": sp["hss_nflops"], "ms": acc["ms_hss_build"], "GFLOPs": gf,
                                   "frac_of_fp64_peak": gf / 1e3 / FP64_PEAK_TFS,
                                   "unit_note": "HSSPACK's nflops model of the structured RRLU "
                                                "(rrluCauchyEigrow/col and pivot searches); latency bound"}
    if sp["zfill_bytes"]:
        b = sp["zfill_bytes"]
        roof = {"kernel": "k_zfill (the zero part of the reordered eigenvector matrix, written on a second "
                          "stream beside the DC levels)",
                "bound": "hbm", "achieved": rate(b, acc["ms_zfill"]), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": rate(b, acc["ms_zfill"]) / HBM_PEAK_GBS,
                "traffic": K_ZFILL_TRAFFIC.get((cfg, n, seed)), "bytes_per_launch": b, "avg_ms": acc["ms_zfill"],
                "timed_in": "profiled pass of %d solves (direct launches, HIP events on the fill's stream)" % nprof,
                "final": {"kernel": "k_final (eigenvector reordering, mdlaed0.f90:355-362: the supported rows)",
                          "bytes_per_launch": sp["final_bytes"], "avg_ms": acc["ms_final"],
                          "achieved": rate(sp["final_bytes"], acc["ms_final"])}}
    else:
        g = rate(sp["final_bytes"], acc["ms_final"])
        roof = {"kernel": "k_final", "bound": "hbm", "achieved": g, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": g / HBM_PEAK_GBS, "traffic": None, "bytes_per_launch": sp["final_bytes"],
                "avg_ms": acc["ms_final"]}
    # ablations
    ctx.set_params(learned=0)
    step()
    classical = timed(3)
    sec_classical = secstats(ctx.stats())
    ctx.set_params(learned=1)
    log("classical start: %.2f ms/solve %s" % (classical * 1e3, sec_classical))
    sync_s = None
    if sync_ablation:
        ctx.set_params(level_sync=1)
        step()
        sync_s = timed(3)
        ctx.set_params(level_sync=0)
        log("host round trip per level: %.2f ms/solve" % (sync_s * 1e3))
    plain_s = None
    if plain:
        ctx.set_params(batched=0, learned=0)
        step()
        plain_s = timed(1)
        ctx.set_params(batched=1, learned=1)
        log("plain (merge at a time, classical start): %.2f ms/solve" % (plain_s * 1e3))
    step()
    torch.cuda.synchronize()
    orth = res = None
    if check:
        orth, res = check_result(torch, d, e, D.cpu().numpy(), Z)
        log("orthogonality %.3e residual %.3e" % (orth, res))
    out = {"value_s": value,
           "schedule": "batched (one launch per DC level, whole solve queued, launch sizes and tables derived "
                       "on the device, HIP graph replay) + learned secular start",
           "profiled_pass_s": t_prof, "batched_classical_s": classical, "batched_level_sync_s": sync_s,
           "plain_s": plain_s, "speedup_vs_plain": plain_s / value if plain_s else None,
           "secular_learned": sec_learned, "secular_classical": sec_classical,
           "iterations_saved_per_root": sec_classical["iters_per_root"] - sec_learned["iters_per_root"],
           "orthogonality": orth, "residual": res,
           "meets_1e12": bool(orth <= 1e-12 and res <= 1e-12) if check else None,
           "merges": int(len(tr["k"])), "levels": st["levels"], "k_top": int(tr["k"][-1]) if len(tr["k"]) else 0,
           "roots": st["roots"], "deflated": st["deflated"], "rotations": int(tr["nrot"].sum()),
           "hss_merges": int(tr["hss"].sum()), "hss_rank_max": int(tr["hss_rank"].max()) if len(tr["k"]) else 0,
           "hot_path_kernels": hot, "roofline": roof}
    del Z
    torch.cuda.empty_cache()
    if h2h:
        # host arrays in and out (MDSTEDC's own interface): the D2H copy of Z is included
        zh = np.zeros((n, n), order="F")
        work, iwork = np.zeros(4), np.zeros(1, np.int32)
        lwork, liwork = 1 + 4 * n + n * n, 3 + 5 * n
        ts = []
        for _ in range(2):
            dh, eh = np.array(d), np.array(e)
            t0 = time.perf_counter()
            info = hsdc.lib().hsdc_stedc(ctx._h, ctypes.c_char(b"I"), n, hsdc._dp(dh), hsdc._dp(eh), hsdc._dp(zh),
                                         n, hsdc._dp(work), lwork, hsdc._ip(iwork), liwork)
            ts.append(time.perf_counter() - t0)
            if info != 0:
                raise RuntimeError("hsdc_stedc returned %d" % info)
        out["host_to_host_s"] = ts[-1]
        log("host to host (hsdc_stedc, Z copied back): %.3f s" % ts[-1])
        del zh
    ctx.close()
    return out


def bench_hss_workload(args, np, torch, hsdc):
    """The near-Toeplitz generator at n = 32768 (d = 2 + U(-1e-3, 1e-3), e = 1 + U(-1e-3, 1e-3),
    seed 4): K close to N at every level, 63 HSS merges.  At HSS tolerance 1e-15 (which meets
    orthogonality and residual <= 1e-12) and 1e-13 (which does not on this matrix)."""
    from hsspack_amd.workloads import tridiag_cfg
    n = 32768
    d, e = tridiag_cfg(1, n, 4)
    out = {"workload": "tridiagonal DC eigensolve, n=%d, %s seed 4, HSS leaf 128, HSS for K>=1024, all "
                       "eigenpairs, device resident" % (n, GEN[1])}
    for tol in (1e-15, 1e-13):
        r = bench_tridiag(args, np, torch, hsdc, 1, n, 4, tol, d, e, 3, 1, plain=(tol == 1e-15), check=True,
                          sync_ablation=False, h2h=False)
        r.pop("roofline")
        out["tol_%g" % tol] = r
    if not args.no_cpu:
        out["cpu_baseline"] = cpu_baseline(1, 4, (1024, 128, 1e-15), n)
        out["cpu_lapack_dstedc"] = cpu_lapack(1, 4, n)
    return out


def bench_batch(args, np, torch, hsdc):
    """512 problems in one batched solve (one launch per DC level over all merges of all problems)
    against a loop of single-problem solves of the same problems."""
    from hsspack_amd.workloads import batch_problems
    probs = batch_problems(512, 256, 8192, 3, cfg=1)
    ns = [len(d) for d, _ in probs]
    offs = np.concatenate([[0], np.cumsum(ns)[:-1]]).astype(np.int64)
    sq = [n * n for n in ns]
    zoffs = np.concatenate([[0], np.cumsum(sq)[:-1]]).astype(np.int64)
    dev = torch.device("cuda:0")
    D0 = torch.tensor(np.concatenate([d for d, _ in probs]), device=dev)
    E0 = torch.tensor(np.concatenate([np.append(e, 0.0) for _, e in probs]), device=dev)
    D, E = torch.empty_like(D0), torch.empty_like(E0)
    Z = torch.empty(int(sum(sq)), dtype=torch.float64, device=dev)
    hss = (1024, 128, args.tol)
    ctx = hsdc.Context(hss_min_k=hss[0], hss_leaf=hss[1], hss_tol=hss[2], batched=1, learned=1)
    ctx.mlp_load(os.path.join(ROOT, "hsspack_amd", "data", "secular_mlp.bin"))
    D.copy_(D0)
    E.copy_(E0)
    leaf, smls, ttimes = ctx.autotune(ns, offs, D, E, Z, zoffs)
    log("autotune: HSS leaf %d, smlsiz %d, candidate ms %s" % (leaf, smls, list(np.round(ttimes, 1))))

    def batched():
        D.copy_(D0)
        E.copy_(E0)
        rc = ctx.stedc_batched_dev(ns, offs, D, E, Z, zoffs)
        if rc != 0:
            raise RuntimeError("hsdc_stedc_batched_dev returned %d" % rc)

    for _ in range(args.warmup):
        batched()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        batched()
    torch.cuda.synchronize()
    t_batch = (time.perf_counter() - t0) / args.steps
    st = ctx.stats()
    log("batched: %.1f ms, stats %s" % (t_batch * 1e3, st))
    # loop of single-problem solves (each with its own per-level launches)
    D.copy_(D0)
    E.copy_(E0)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for k, n in enumerate(ns):
        o, zo = int(offs[k]), int(zoffs[k])
        rc = ctx.stedc_dev(D[o:o + n], E[o:o + n], Z[zo:zo + n * n].view(n, n))
        if rc != 0:
            raise RuntimeError("hsdc_stedc_dev returned %d" % rc)
    torch.cuda.synchronize()
    t_loop = time.perf_counter() - t0
    log("loop of single solves: %.1f ms" % (t_loop * 1e3))
    batched()
    torch.cuda.synchronize()
    # orthogonality and residual of every 32nd problem
    worst = [0.0, 0.0]
    Dh = D.cpu().numpy()
    for k in range(0, len(ns), 32):
        n, o, zo = ns[k], int(offs[k]), int(zoffs[k])
        d, e = probs[k]
        orth, res = check_result(torch, d, e, Dh[o:o + n], Z[zo:zo + n * n].view(n, n))
        worst = [max(worst[0], orth), max(worst[1], res)]
    log("checked problems: orthogonality %.3e residual %.3e" % tuple(worst))
    print(json.dumps({
        "metric": "s to all eigenpairs of 512 tridiagonals (n log-uniform in [256, 8192]): batched vs loop",
        "value": t_batch, "unit": "s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": t_batch * 1e3, "higher_is_better": False, "scaling": "weak", "vs_baseline": None,
        "dtype": "f64", "data": "synthetic",
        "config": {"workload": "512 tridiagonals, n log-uniform in [256, 8192] seed 3, d=2+U(-1e-3,1e-3), "
                               "e=1+U(-1e-3,1e-3), HSS for K>=1024, autotuned leaves, tol %g, device resident"
                               % hss[2],
                   "total_n": int(sum(ns)), "loop_s": t_loop, "speedup_vs_loop": t_loop / t_batch,
                   "levels": st["levels"], "merges": st["merges"], "hss_merges": st["hss_merges"],
                   "autotuned": {"hss_leaf": leaf, "smlsiz": smls,
                                 "candidates_ms": {"smlsiz %d leaf %d" % (a, b): float(ttimes[3 * i + j])
                                                   for i, a in enumerate((25, 40))
                                                   for j, b in enumerate((64, 128, 256))}},
                   "orthogonality_worst_of_16": worst[0], "residual_worst_of_16": worst[1]}}), flush=True)


def bench_svd(args, np, torch, hsdc):
    """Bidiagonal SVD workload: all singular triplets of the order-16384 upper bidiagonal
    d ~ U(0.5, 1.5), e ~ U(0, 1) (seed 5), device resident, through hsdc_bdsdc_dev.
    With --svd-toeplitz the near-Toeplitz bidiagonal (1 + 1e-3 N(0,1), seed 11), whose
    large merges take the HSS branch; the same matrix with the dense branch only is
    timed beside it."""
    from hsspack_amd.workloads import bidiag_cfg, bidiag_toeplitz
    n = args.n if args.n != 32768 else 16384
    toep = args.svd_toeplitz
    d, e = bidiag_toeplitz(n, 11) if toep else bidiag_cfg(n, seed=5)
    dev = torch.device("cuda:0")
    D0 = torch.tensor(d, device=dev)
    E0 = torch.tensor(e, device=dev)
    D, E = torch.empty_like(D0), torch.empty_like(E0)
    U = torch.empty((n, n), dtype=torch.float64, device=dev)
    VT = torch.empty((n, n), dtype=torch.float64, device=dev)
    # HSS leaf 128 for the near-Toeplitz workload: measured 126 ms against 180 ms with the
    # reference's Ni = 40 (the ranks, 60-97, do not shrink with the leaf, so larger
    # leaves mean fewer tree levels of intermediate products); threshold 2000 as in the
    # reference (1024 and 512 measured slower)
    hss_leaf = args.hss_leaf or (128 if toep else 40)
    ctx = hsdc.BdContext(hss_leaf=hss_leaf, hss_min_k=args.hss_min_k)

    def step():
        D.copy_(D0)
        E.copy_(E0)
        rc = ctx.bdsdc_dev(D, E, U, VT)
        if rc != 0:
            raise RuntimeError("hsdc_bdsdc_dev returned %d" % rc)

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    t = (time.perf_counter() - t0) / args.steps
    st = ctx.stats()
    log("bdsdc n=%d: %.2f ms, stats %s" % (n, t * 1e3, st))
    out = {}
    if toep:
        out.update(hss_merges=st["hss_merges"], hss_rank_max=st["hss_rank_max"])
        if not args.no_plain:
            # the same matrix with every merge on the dense branch (DLASD3)
            ctx.set_params(hss_min_k=n + 1)
            step()
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(2):
                step()
            torch.cuda.synchronize()
            td = (time.perf_counter() - t0) / 2
            ctx.set_params(hss_min_k=args.hss_min_k)
            step()
            torch.cuda.synchronize()
            out.update(dense_only_s=td, speedup_vs_dense=td / t)
            log("dense branch only: %.2f ms (HSS branch %.2fx faster)" % (td * 1e3, td / t))
    if not args.no_check:
        I = torch.eye(n, dtype=torch.float64, device=dev)
        Uc, Vc = U.t(), VT.t()
        orth_u = (Uc.t() @ Uc - I).abs().max().item()
        orth_v = (Vc @ Vc.t() - I).abs().max().item()
        del I
        B = torch.zeros((n, n), dtype=torch.float64, device=dev)
        idx = torch.arange(n, device=dev)
        B[idx, idx] = D0
        B[idx[:-1], idx[1:]] = E0
        res = ((Uc * D) @ Vc - B).abs().max().item() / B.abs().max().item()
        del B
        s = D.cpu().numpy()
        out.update(orthogonality_u=orth_u, orthogonality_v=orth_v, residual=res,
                   sorted_descending=bool(np.all(np.diff(s) <= 0)))
        log("orthogonality U %.2e V %.2e residual %.2e" % (orth_u, orth_v, res))
    cpu = None
    if not args.no_cpu and not toep:
        sys.path.insert(0, os.path.join(ROOT, "tests"))
        import oracle_py as O
        times = {}
        for m in (4096, 8192):
            dm, em = bidiag_cfg(m, seed=5)
            t0 = time.perf_counter()
            r = O.bdsdc(dm, em)
            times[m] = time.perf_counter() - t0
            assert r["info"] == 0
            log("cpu oracle bdsdc n=%d: %.2f s" % (m, times[m]))
        p = np.log2(times[8192] / times[4096])
        est = times[8192] * (n / 8192.0) ** p
        cpu = dict(value=est, unit="s", cores=1, kind="port",
                   sample="oracle (C restatement of mdbdsdc/mdlasd0-2 + DLASD3/DLASD4, 1 thread) on the "
                          "same generator at n=4096 (%.2f s) and n=8192 (%.2f s), extrapolated to n=%d with "
                          "the measured exponent %.2f" % (times[4096], times[8192], n, p))
    print(json.dumps({
        "metric": "s to all singular triplets, n=%d FP64 upper bidiagonal (orth<=1e-12)" % n,
        "value": t, "unit": "s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": t * 1e3, "higher_is_better": False, "scaling": "weak", "vs_baseline": None,
        "dtype": "f64", "data": "synthetic",
        "config": dict({"workload": ("upper bidiagonal n=%d, d,e = 1+1e-3 N(0,1) seed 11 (near-Toeplitz), "
                                     "leaf 25, HSS branch for K>=%d (HSS leaf %d, tol 1e-17), all singular "
                                     "triplets, device resident" % (n, args.hss_min_k, hss_leaf)) if toep else
                                    ("upper bidiagonal n=%d, d=U(0.5,1.5), e=U(0,1) seed 5, leaf 25, all "
                                     "singular triplets, device resident" % n),
                        "levels": st["levels"], "merges": st["merges"], "roots": st["roots"],
                        "deflated": st["deflated"], "rotations": st["rotations"], "k_top": st["k_top"],
                        "iters_per_root": st["secular_iters"] / max(st["roots"], 1),
                        "ms_device": st["ms_total"]}, **out),
        "cpu_baseline": cpu}), flush=True)


def bench_band(args, np, torch, hsdc):
    """Banded workload: all eigenpairs of the order-16384 symmetric band matrix with
    KD = 64 and N(0,1) entries (seed 6), device resident, through hsdc_sbevd_dev:
    leaves of 128 rows, the HSS branch for updates with K >= 1500 (HSS leaf 128,
    tolerance 1e-17).  Also: a profiled pass (HSS construction and multiply rates), the
    dense-branch-only ablation, orthogonality and residual, the oracle at n = 1024 and
    2048 extrapolated, and LAPACK dsbevd (scipy eig_banded) on the host's threads."""
    from hsspack_amd.workloads import band_cfg
    n = args.n if args.n != 32768 else 16384
    kd = args.kd
    ab = band_cfg(n, kd, seed=6, sub=0)
    dev = torch.device("cuda:0")
    abt = torch.tensor(np.ascontiguousarray(ab.T), device=dev)
    w = torch.empty(n, dtype=torch.float64, device=dev)
    q = torch.empty((n, n), dtype=torch.float64, device=dev)
    hss_leaf = args.hss_leaf or 128
    hmin = args.hss_min_k if args.hss_min_k != 2000 else 1500
    ctx = hsdc.SbContext(hss_min_k=hmin, hss_leaf=hss_leaf, hss_tol=1e-17)

    def step():
        rc = ctx.sbevd_dev(abt, kd, w, q)
        if rc != 0:
            raise RuntimeError("hsdc_sbevd_dev returned %d" % rc)

    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    t = (time.perf_counter() - t0) / args.steps
    st = ctx.stats()
    log("sbevd n=%d kd=%d: %.1f ms, stats %s" % (n, kd, t * 1e3, st))
    # profiled pass: event-timed HSS phases
    ctx.set_params(profile=1)
    step()
    torch.cuda.synchronize()
    sp = ctx.stats()
    ctx.set_params(profile=0)
    out = dict(levels=st["levels"], leaves=st["leaves"], updates=st["updates"], roots=st["roots"],
               deflated=st["deflated"], rotations=st["rotations"], hss_updates=st["hss_updates"],
               hss_rank_max=st["hss_rank_max"], iters_per_root=st["secular_iters"] / max(st["roots"], 1),
               ms_device=st["ms_total"], dense_tflop=st["dense_flops"] / 1e12)
    build_rate = sp["hss_nflops"] / (sp["ms_hss_build"] * 1e-3) / 1e12 if sp["ms_hss_build"] > 0 else None
    mm_rate = sp["hss_mm_flops"] / (sp["ms_hss_mm"] * 1e-3) / 1e12 if sp["ms_hss_mm"] > 0 else None
    out["hss_construction"] = dict(ms=sp["ms_hss_build"], model_tflop=sp["hss_nflops"] / 1e12,
                                   tflops_in_model=build_rate, frac_fp64_peak=(build_rate or 0) / FP64_PEAK_TFS,
                                   share_of_solve=sp["ms_hss_build"] / sp["ms_total"])
    out["hss_multiply"] = dict(ms=sp["ms_hss_mm"], tflop=sp["hss_mm_flops"] / 1e12, tflops=mm_rate,
                               frac_fp64_peak=(mm_rate or 0) / FP64_PEAK_TFS)
    roof = {"bound": "mfma", "kernel": "HSS construction (k_hss_rowcomp + k_hss_colcomp), the largest share",
            "achieved": build_rate, "peak": FP64_PEAK_TFS, "unit": "TFLOP/s",
            "frac": (build_rate or 0) / FP64_PEAK_TFS, "traffic": None,
            "note": "flops in HSSPACK's RRLU model over the event-timed construction; the structured "
                    "RRLU is a chain of dependent pivot steps per HSS node, so the rate is latency-bound"}
    if not args.no_plain:
        ctx.set_params(hss_min_k=0)
        step()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        step()
        torch.cuda.synchronize()
        td = time.perf_counter() - t0
        sd = ctx.stats()
        ctx.set_params(hss_min_k=hmin)
        out.update(dense_only_s=td, dense_only_tflop=sd["dense_flops"] / 1e12,
                   dense_only_tflops=sd["dense_flops"] / td / 1e12, speedup_vs_dense=td / t)
        log("dense branch only: %.1f ms (%.1f TFLOP, %.1f TF/s)" % (td * 1e3, sd["dense_flops"] / 1e12,
                                                                  sd["dense_flops"] / td / 1e12))
    if not args.no_check:
        A = torch.zeros((n, n), dtype=torch.float64, device=dev)
        abd = torch.tensor(ab, device=dev)
        j = torch.arange(n, device=dev)
        for r in range(kd + 1):
            off = kd - r
            jj = j[off:]
            A[jj - off, jj] = abd[r, off:]
            A[jj, jj - off] = abd[r, off:]
        Q = q.t()
        orth = res = 0.0
        for i0 in range(0, n, 4096):
            g = Q[:, i0:i0 + 4096].t() @ Q
            g[:, i0:i0 + 4096].diagonal().sub_(1.0)
            orth = max(orth, g.abs().max().item())
            del g
            rr = A @ Q[:, i0:i0 + 4096] - Q[:, i0:i0 + 4096] * w[i0:i0 + 4096]
            res = max(res, rr.abs().max().item())
            del rr
        res /= A.abs().max().item()
        del A
        out.update(orthogonality=orth, residual=res)
        log("orthogonality %.2e residual %.2e" % (orth, res))
    cpu = None
    if not args.no_cpu:
        sys.path.insert(0, os.path.join(ROOT, "tests"))
        import oracle_py as O
        import scipy.linalg as sl
        times = {}
        for m in (1024, 2048):
            abm = band_cfg(m, kd, seed=6, sub=0)
            t0 = time.perf_counter()
            r = O.sbevd(abm, kd, smlsiz=128)
            times[m] = time.perf_counter() - t0
            assert r["info"] == 0
            log("cpu oracle sbevd n=%d: %.2f s (%d threads)" % (m, times[m], host_threads()))
        est, p = _extrapolate(np, times, n)
        cpu = dict(value=est, unit="s", cores=host_threads(), cpu=cpu_model(), kind="port",
                   sample="oracle (C restatement of mdsbevd/mdsbed1 with dense secular vectors, OpenMP over "
                          "independent GEMM columns) on the same generator at n=1024 (%.2f s) and n=2048 (%.2f s), "
                          "extrapolated to n=%d with the measured exponent %.2f" % (times[1024], times[2048], n, p))
        lt = {}
        for m in (4096, 8192):
            abm = band_cfg(m, kd, seed=6, sub=0)
            t0 = time.perf_counter()
            sl.eig_banded(abm, lower=False)
            lt[m] = time.perf_counter() - t0
            log("cpu LAPACK eig_banded n=%d: %.2f s" % (m, lt[m]))
        le, lp = _extrapolate(np, lt, n)
        out["cpu_lapack_dsbevd"] = dict(value=le, unit="s", cores=host_threads(), kind="lapack",
                                        sample="scipy eig_banded (LAPACK band reduction + tridiagonal solve, "
                                               "OpenBLAS) at n=4096 (%.2f s) and 8192 (%.2f s), extrapolated "
                                               "with exponent %.2f" % (lt[4096], lt[8192], lp))
    print(json.dumps({
        "metric": "s to all eigenpairs, n=%d FP64 symmetric band KD=%d (MDSBEVD path)" % (n, kd),
        "value": t, "unit": "s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": t * 1e3, "higher_is_better": False, "scaling": "weak", "vs_baseline": None,
        "dtype": "f64", "data": "synthetic",
        "config": dict({"workload": "symmetric band n=%d KD=%d, N(0,1) entries seed 6, leaves 128, HSS branch "
                                    "for K>=%d (HSS leaf %d, tol 1e-17), all eigenpairs, device resident"
                                    % (n, kd, hmin, hss_leaf)}, **out),
        "roofline": roof, "cpu_baseline": cpu}, default=lambda o: o.item() if hasattr(o, "item") else str(o)),
        flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--n", type=int, default=32768)
    ap.add_argument("--cfg", type=int, default=2)
    ap.add_argument("--seed", type=int, default=2)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-plain", action="store_true")
    ap.add_argument("--no-check", action="store_true")
    ap.add_argument("--no-hss", action="store_true", help="skip the n=32768 near-Toeplitz (HSS) sub-record")
    ap.add_argument("--tol", type=float, default=1e-13, help="HSS compression tolerance")
    ap.add_argument("--batch", action="store_true",
                    help="512 independent tridiagonals, n log-uniform in [256, 8192] (near-Toeplitz entries, "
                         "seed 3): one batched solve against a loop of single-problem solves")
    ap.add_argument("--svd", action="store_true",
                    help="bidiagonal SVD: all singular triplets of the order-16384 upper bidiagonal "
                         "d=U(0.5,1.5), e=U(0,1), seed 5 (MDBDSDC path)")
    ap.add_argument("--svd-toeplitz", action="store_true",
                    help="with --svd: the near-Toeplitz bidiagonal (HSS branch at the top merges), "
                         "timed against the dense branch alone")
    ap.add_argument("--band", action="store_true",
                    help="banded DC: all eigenpairs of the order-16384 symmetric band matrix, KD=64, N(0,1) "
                         "entries, seed 6 (MDSBEVD path)")
    ap.add_argument("--kd", type=int, default=64, help="with --band: the bandwidth")
    ap.add_argument("--hss-leaf", type=int, default=0,
                    help="with --svd / --band: HSS leaf block (default 128 with --svd-toeplitz and --band, else 40)")
    ap.add_argument("--hss-min-k", type=int, default=2000,
                    help="with --svd / --band: a merge (update) with K >= this takes the HSS branch (default "
                         "2000; 1500 with --band)")
    ap.add_argument("--copy-probe", action="store_true",
                    help="only copy 1 GiB device to device three times (calibrates rocprofv3 byte counters)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU only: the solver runs on a single MI355X and has no "
              "multi-GPU path; run with --gpus 1", file=sys.stderr)
        sys.exit(2)
    import numpy as np
    import torch
    if args.copy_probe:
        src = torch.ones(1 << 27, dtype=torch.float64, device="cuda:0")
        dst = torch.empty_like(src)
        e0, e1, e2 = (torch.cuda.Event(enable_timing=True) for _ in range(3))
        for _ in range(3):
            dst.copy_(src)
        e0.record()
        for _ in range(5):
            dst.copy_(src)
        e1.record()
        for _ in range(5):
            dst.fill_(0.0)
        e2.record()
        torch.cuda.synchronize()
        nb = src.numel() * 8
        print(json.dumps({"copy_probe_bytes": nb,
                          "copy_GBps": 2 * nb * 5 / (e0.elapsed_time(e1) * 1e-3) / 1e9,
                          "fill_GBps": nb * 5 / (e1.elapsed_time(e2) * 1e-3) / 1e9}))
        return
    from hsspack_amd import hsdc
    from hsspack_amd.workloads import tridiag_cfg
    if args.batch:
        return bench_batch(args, np, torch, hsdc)
    if args.svd:
        return bench_svd(args, np, torch, hsdc)
    if args.band:
        return bench_band(args, np, torch, hsdc)

    n = args.n
    d, e = tridiag_cfg(args.cfg, n, args.seed)
    r = bench_tridiag(args, np, torch, hsdc, args.cfg, n, args.seed, args.tol, d, e, args.steps, args.warmup,
                      plain=not args.no_plain, check=not args.no_check, sync_ablation=True)
    roof = r.pop("roofline")
    out = {
        "metric": "s to all eigenpairs, n=32768 FP64 tridiag (orth<=1e-12): learned+batched vs plain",
        "value": r["value_s"],
        "unit": "s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": r["value_s"] * 1e3,
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": dict({"workload": "tridiagonal DC eigensolve, n=%d, %s seed %d, HSS leaf 128, tol %g, HSS for "
                                    "K>=1024, all eigenpairs, device resident" % (n, GEN[args.cfg], args.seed,
                                                                                   args.tol),
                        "n": n}, **{k: v for k, v in r.items() if k != "value_s"}),
        "roofline": roof,
    }
    if not args.no_hss:
        out["config"]["hss_workload"] = bench_hss_workload(args, np, torch, hsdc)
    if not args.no_cpu:
        out["cpu_baseline"] = cpu_baseline(args.cfg, args.seed, (1024, 128, args.tol), n)
        out["config"]["cpu_lapack_dstedc"] = cpu_lapack(args.cfg, args.seed, n)
        gpu_h2h = out["config"].get("host_to_host_s")
        if gpu_h2h:
            out["config"]["gpu_host_to_host_vs_cpu"] = {
                "vs_oracle": out["cpu_baseline"]["value"] / gpu_h2h,
                "vs_lapack_dstedc": out["config"]["cpu_lapack_dstedc"]["value"] / gpu_h2h}
    print(json.dumps(out, default=lambda o: o.item() if hasattr(o, "item") else str(o)), flush=True)

if __name__ == "__main__":
    main()
