#!/usr/bin/env python3
"""Headline benchmark: LU-solve TFLOP/s, FP32-MFMA + iterative refinement vs
plain FP64, at a normwise backward error <= 1e-12; DGEMM % of FP64 peak.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--only SECTION]

One step = one mixed-precision solve x = b/A of the mixed-precision
configuration: A = U diag(s) V^T, n = 16384, U and V orthogonal factors of
seeded Gaussian matrices (QR), s log-spaced from 1 to 1/kappa (kappa =
1e4), b ~ N(0,1), 1 right-hand side; FP32 LU with partial pivoting on MFMA,
FP64 residual and update on the GPU until backward error <= 1e-12.
`value` = effective FP64-equivalent TFLOP/s, ((2/3) n^3 + 2 n^2) / time per
solve (the HPL-MxP convention), inputs resident in HBM.

Also measured in the same run (outside the K timed steps):
  - `roofline_step`: the dominant kernel of the step, the FP32 panel
    factorisation (panel_kernel<float>), timed with HIP events on the
    stream it runs on during one more solve; algorithmic bytes = the panel
    read once and written once (8 m jb bytes for an m x jb FP32 panel);
  - the mixed solver over kappa in {1e2, 1e4, 1e6}: FP32 factorisation
    with 1 and 64 right-hand sides, FP16 and BF16 trailing updates with
    GMRES-IR, each against the plain FP64 GPU LU solve on the same A and b;
  - the plain-FP64 configurations: DGEMM M = N = K = 8192 in the CCC, CRC
    and RCC operand layouts (CCC is the `roofline` entry, FP64 MFMA,
    78.6 TFLOP/s peak, HIP events on the stream it runs on) and the FP64
    LU n = 8192 with 16 right-hand sides (uniform[-1,1], b ~ N(0,1));
    the CPU-sized case: DGEMM 512^3 and the LU solve n = 512 (A + n I);
  - the batched workload: 20,000 systems n ~ U{8..128} (+ n on the
    diagonal), nrhs ~ U{1..4}, FP64 and FP32, factor + solve in one
    hipGraph replay (three launches) vs per-matrix
    launches, plus the batched GEMM with K = n;
  - the differentiation workload: 512 systems n = 256, forward solve and
    the adjoint (grad_b = A^-T g, grad_A = -grad_b x^T) with stored and
    with recomputed factors;
  - the CPU baseline: the real TMV 0.76 library (oracle/_ref, built from
    the reference sources) on the host's cores (OpenMP), best of 3 with a
    cache flush between runs: x = b/A at n = 4096 (the bounded sample of
    the headline workload, `cpu_baseline`), and the 512 case (GEMM and LU
    solve); --cpu-cfg2 adds the 8192 case (three GEMM layouts, LU + 16
    right-hand sides; minutes of CPU time).  The oracle restatement (kind
    "port") stands in where the TMV build is absent.
--only mixed|fp64|batched|cpu runs one section (profiling); the JSON line
then carries that section's figures only.
Prints ONE JSON line.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_FP64_TFLOPS = 78.6
PEAK_FP32_TFLOPS = 157.3
PEAK_HBM_GBS = 8000.0
SEED = 0x7A15EED
# HBM bytes per launch of the 8192^3 CCC DGEMM (gemm_kernel f64 128x128x16),
# from rocprofv3 --pmc FETCH_SIZE (x2.0) and WRITE_SIZE (x1.0), the factors a
# 1 GiB device copy reads on the same counters; profiles/dgemm_8192_ccc_traffic.md.
DGEMM_8192_CCC_TRAFFIC = 13.43e9
# HBM bytes per launch of the FP32 panel kernel (64-column panels), averaged
# over the 256 panels of an n = 16384 LU (same counters and factors);
# profiles/panel_f32_n16384_traffic.md.
PANEL_F32_16384_TRAFFIC = {64: 6.40e6}


def conditioned_gpu(n, kappa, seed, torch, tmv_amd):
    """A = U diag(s) V^T (column-major FP64 on the GPU)."""
    g = torch.empty(n * n, dtype=torch.float64, device="cuda")
    tmv_amd.fill_normal(g, seed)
    U, _ = torch.linalg.qr(g.view(n, n))
    tmv_amd.fill_normal(g, seed + 1)
    V, _ = torch.linalg.qr(g.view(n, n))
    del g
    s = torch.logspace(0, -torch.log10(torch.tensor(kappa)).item(), n,
                       dtype=torch.float64, device="cuda")
    US = (U * s[None, :]).contiguous()          # row-major storage of U diag(s)
    del U
    A = tmv_amd.gemm(US, V.t())                 # column-major U diag(s) V^T
    del US, V
    torch.cuda.empty_cache()
    return A


def backward_error_gpu(A, x, b, torch):
    """max over columns of ||b - A x||_inf / (||A||_inf ||x||_inf + ||b||_inf)."""
    X = x if x.dim() > 1 else x.view(-1, 1)
    B = b if b.dim() > 1 else b.view(-1, 1)
    r = B - A @ X
    nA = A.abs().sum(dim=1).max()
    be = r.abs().max(dim=0).values / (nA * X.abs().max(dim=0).values + B.abs().max(dim=0).values)
    return float(be.max())


def _flush_cache(np, buf=[None]):
    """Touch 256 MiB so that the next CPU run starts from cold caches (as
    TMV's speed harness does between runs)."""
    if buf[0] is None:
        buf[0] = np.ones(32 << 20)
    buf[0] += 1.0


def _best_of(np, fn, reps, cap_s):
    best = None
    t_start = time.perf_counter()
    for _ in range(reps):
        _flush_cache(np)
        t0 = time.perf_counter()
        fn()
        dt = time.perf_counter() - t0
        best = dt if best is None else min(best, dt)
        if time.perf_counter() - t_start > cap_s:
            break
    return best


def _progress(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def _cpu_lib():
    import oracle
    lib = oracle.ref_lib()
    if lib is None:
        oracle.build()
    return oracle, lib, ("reference" if lib is not None else "port")


def cpu_baseline(seconds_cap=30.0):
    """TMV's own CPU path on a bounded sample of the headline workload:
    x = b/A, n = 4096, best of 3."""
    import numpy as np
    from tmv_amd import rng
    oracle, lib, kind = _cpu_lib()
    n = 4096
    A = rng.uniform_matrix(SEED + 4000, n, n)
    b = rng.uniform(SEED + 4001, n, -1.0, 1.0)
    solve = (lambda: oracle.ref_gesv(A, b)) if lib is not None else (lambda: oracle.gesv(A, b))
    best = _best_of(np, solve, 3, seconds_cap)
    flops = 2.0 / 3.0 * n ** 3 + 2.0 * n * n
    threads = (lib or oracle.oracle_lib()).fn("num_threads")()
    return {"value": round(flops / best / 1e12, 5), "unit": "TFLOP/s", "cores": int(threads),
            "kind": kind,
            "sample": (f"x = b/A (divideUsing LU: LU_Decompose + LU_LDivEq, OpenMP MultMM), "
                       f"n={n}, uniform[-1,1] seeded, best of 3, {best * 1e3:.0f} ms"),
            "ms": round(best * 1e3, 1)}


def cpu_configs(cfg2=False, reps=3):
    """TMV on the plain-FP64 configurations: DGEMM 512^3 and the LU solve
    n = 512 (A + n I, 1 right-hand side); with cfg2 also DGEMM 8192^3 in
    the CCC, CRC and RCC layouts and the LU n = 8192 with 16 right-hand
    sides.  Best of `reps` (each run capped in total time), cache flushed
    between runs."""
    import numpy as np
    from tmv_amd import rng
    oracle, lib, kind = _cpu_lib()
    threads = int((lib or oracle.oracle_lib()).fn("num_threads")())
    out = {"kind": kind, "cores": threads, "reps": reps}
    gesv = oracle.ref_gesv if lib is not None else oracle.gesv

    n = 512
    A = np.asfortranarray(rng.uniform_matrix(SEED + 100, n, n))
    B = np.asfortranarray(rng.uniform_matrix(SEED + 101, n, n))
    t = _best_of(np, lambda: oracle.gemm(A, B, lib=lib), reps, 20.0)
    out["dgemm_512"] = {"us": round(t * 1e6, 1), "gflops": round(2 * n ** 3 / t / 1e9, 2)}
    A = A + n * np.eye(n)
    b = rng.uniform(SEED + 102, n, -1.0, 1.0)
    t = _best_of(np, lambda: gesv(A, b), reps, 20.0)
    out["lu_solve_512"] = {"us": round(t * 1e6, 1),
                           "gflops": round((2 / 3 * n ** 3 + 2 * n * n) / t / 1e9, 2)}
    if cfg2:
        n = 8192
        Ac = np.asfortranarray(rng.uniform_matrix(SEED + 200, n, n))
        Bc = np.asfortranarray(rng.uniform_matrix(SEED + 201, n, n))
        Ar = np.ascontiguousarray(Ac)
        Br = np.ascontiguousarray(Bc)
        for name, a_, b_, arm, brm in (("CCC", Ac, Bc, False, False),
                                       ("CRC", Ar, Bc, True, False),
                                       ("RCC", Ac, Br, False, True)):
            _progress(f"TMV DGEMM 8192 {name}")
            t = _best_of(np, lambda: oracle.gemm(a_, b_, a_rowmajor=arm, b_rowmajor=brm, lib=lib),
                         reps, 60.0)
            out[f"dgemm_8192_{name}"] = {"s": round(t, 3), "gflops": round(2 * n ** 3 / t / 1e9, 2)}
        del Ar, Br, Bc
        Bn = np.asfortranarray(np.random.default_rng(SEED + 202).standard_normal((n, 16)))
        _progress("TMV LU 8192, 16 RHS")
        t = _best_of(np, lambda: gesv(Ac, Bn), reps, 60.0)
        out["lu_8192_nrhs16"] = {"s": round(t, 3),
                                 "gflops": round((2 / 3 * n ** 3 + 2 * n * n * 16) / t / 1e9, 2)}
    return out


def batched_workload(torch, tmv_amd, dtype, count=20000, reps=5, per_matrix_sample=200):
    """20,000 independent systems, n ~ U{8..128}, entries uniform[-1,1] + n on
    the diagonal, nrhs ~ U{1..4}: factor + solve in three launches
    replayed from a hipGraph, the batched GEMM C_i = A_i B_i
    with K = n_i, and the same systems through per-matrix launches."""
    import numpy as np
    g = np.random.default_rng(SEED + 30)
    ns = g.integers(8, 129, count).astype(np.int32)
    nrhs = g.integers(1, 5, count).astype(np.int32)
    b = tmv_amd.Batch(ns, nrhs, dtype=dtype)
    tmp = torch.empty(b.A.numel(), dtype=torch.float64, device="cuda")
    tmv_amd.fill_uniform(tmp, SEED + 31)
    diag = np.concatenate([b.offA[i] + np.arange(n) * (n + 1) for i, n in enumerate(ns)])
    dval = np.repeat(ns.astype(np.float64), ns)
    tmp[torch.as_tensor(diag, device="cuda")] += torch.as_tensor(dval, device="cuda")
    A0 = tmp.to(dtype)
    tmp = torch.empty(b.B.numel(), dtype=torch.float64, device="cuda")
    tmv_amd.fill_uniform(tmp, SEED + 32)
    B0 = tmp.to(dtype)
    del tmp
    t0 = time.perf_counter()
    plan = tmv_amd.BatchPlan(b, tune=True)
    tune_s = time.perf_counter() - t0
    s = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    b.A.copy_(A0); b.B.copy_(B0)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=s):
        tmv_amd.gesv_batched(plan, b, stream=s)
    times = []
    for _ in range(reps + 1):
        b.A.copy_(A0); b.B.copy_(B0)
        torch.cuda.synchronize()
        e0 = torch.cuda.Event(enable_timing=True); e1 = torch.cuda.Event(enable_timing=True)
        with torch.cuda.stream(s):
            e0.record(s); graph.replay(); e1.record(s)
        torch.cuda.synchronize()
        times.append(e0.elapsed_time(e1))
    ms = min(times[1:])
    bad = int((b.info != 0).sum().item())
    # solution check on a sample: backward error per column
    worst = 0.0
    for i in range(0, count, max(1, count // 50)):
        n = int(ns[i])
        o = int(b.offA[i])
        Ai = A0[o:o + n * n].view(n, n).t().double()
        X = b.b(i).double()
        ob = int(b.offB[i])
        Bi = B0[ob:ob + n * int(nrhs[i])].view(int(nrhs[i]), n).t().double()
        r = Bi - Ai @ X
        be = (r.abs().max(dim=0).values /
              (Ai.abs().sum(dim=1).max() * X.abs().max(dim=0).values + Bi.abs().max(dim=0).values))
        worst = max(worst, float(be.max()))
    n64 = ns.astype(np.float64)
    flops = float((2.0 / 3.0 * n64 ** 3 + 2.0 * n64 ** 2 * nrhs).sum())
    esz = b.A.element_size()
    bytes_ = float((2 * n64 ** 2 + 2 * n64 * nrhs).sum() * esz + n64.sum() * 8)
    out = {"systems": count, "dtype": str(dtype).replace("torch.", ""), "ms": round(ms, 3),
           "tflops": round(flops / ms / 1e9, 3), "gbs": round(bytes_ / ms / 1e6, 1),
           "hbm_frac": round(bytes_ / ms / 1e6 / 8000.0, 4),
           "singular": bad, "worst_backward_error": worst,
           "plan": plan.describe(), "tune_s": round(tune_s, 2),
           "algorithmic": {"flops": flops, "bytes": bytes_}}
    # per-matrix launches: the same kernel launched once per system (sample)
    k = min(per_matrix_sample * 10, count)
    plans = [tmv_amd.BatchPlan([int(ns[i])], [int(nrhs[i])], dtype=dtype) for i in range(k)]
    singles = [tmv_amd.Batch([int(ns[i])], [int(nrhs[i])], dtype=dtype) for i in range(k)]
    for i in range(k):
        singles[i].A.copy_(A0[int(b.offA[i]):int(b.offA[i]) + int(ns[i]) ** 2])
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    for i in range(k):
        tmv_amd.gesv_batched(plans[i], singles[i])
    torch.cuda.synchronize()
    per_launch = (time.perf_counter() - t1) / k
    del plans, singles
    # per-matrix general path (blocked getrf + getrs, as a TMV caller's loop)
    k2 = min(per_matrix_sample, count)
    Ms = [A0[int(b.offA[i]):int(b.offA[i]) + int(ns[i]) ** 2].view(int(ns[i]), int(ns[i])).t().clone()
          for i in range(k2)]
    Ms = [tmv_amd.colmajor(m) for m in Ms]
    Xs = [torch.ones(int(ns[i]), int(nrhs[i]), dtype=dtype, device="cuda").t().contiguous().t()
          for i in range(k2)]
    torch.cuda.synchronize()
    t2 = time.perf_counter()
    for i in range(k2):
        piv, _ = tmv_amd.getrf(Ms[i])
        tmv_amd.getrs(Ms[i], piv, Xs[i], check_singular=False)
    torch.cuda.synchronize()
    per_general = (time.perf_counter() - t2) / k2
    out["per_matrix_launch_ms"] = round(per_launch * count * 1e3, 2)
    out["per_matrix_launch_sample"] = k
    out["per_matrix_getrf_getrs_ms"] = round(per_general * count * 1e3, 1)
    out["per_matrix_getrf_getrs_sample"] = k2
    out["speedup_vs_per_matrix_launch"] = round(per_launch * count * 1e3 / ms, 1)
    # batched GEMM, K = n: C_i = A_i B_i (A_i and B_i the systems' matrices)
    C = torch.empty_like(b.A)
    pC = torch.as_tensor(C.data_ptr() + esz * b.offA, device="cuda")
    pA0 = torch.as_tensor(A0.data_ptr() + esz * b.offA, device="cuda")
    gt = []
    for _ in range(reps + 1):
        e0 = torch.cuda.Event(enable_timing=True); e1 = torch.cuda.Event(enable_timing=True)
        e0.record()
        tmv_amd.gemm_batched(b.d_n, b.d_n, b.d_n, pA0, pA0, pC, dtype=dtype)
        e1.record()
        torch.cuda.synchronize()
        gt.append(e0.elapsed_time(e1))
    gms = min(gt[1:])
    gflops = float((2.0 * n64 ** 3).sum())
    gbytes = float((3 * n64 ** 2).sum() * esz)
    out["gemm"] = {"ms": round(gms, 3), "tflops": round(gflops / gms / 1e9, 2),
                   "gbs": round(gbytes / gms / 1e6, 1)}
    del b, A0, B0, C, graph
    torch.cuda.empty_cache()
    return out


def adjoint_workload(torch, tmv_amd, dtype, count=512, n=256, reps=3):
    """512 systems, n = 256: A = Q diag(s) Q^T + n I (Q from the QR of a
    seeded Gaussian, s ~ U[0.1, 10]), b, w ~ N(0, 1), loss = sum(w .* x).
    Forward: batched factorisation + solve; backward: the adjoint kernel
    with stored factors, and with recomputed factors."""
    import numpy as np
    ns = np.full(count, n, np.int32)
    nr = np.ones(count, np.int32)
    b = tmv_amd.Batch(ns, nr, dtype=dtype)
    g = torch.empty(n * n, dtype=torch.float64, device="cuda")
    tmv_amd.fill_normal(g, SEED + 50)
    Q, _ = torch.linalg.qr(g.view(n, n))
    s = torch.empty(count * n, dtype=torch.float64, device="cuda")
    tmv_amd.fill_uniform(s, SEED + 51, 0.1, 10.0)
    Qs = Q.unsqueeze(0) * s.view(count, 1, n)                  # Q diag(s_b)
    A3 = torch.matmul(Qs, Q.t().contiguous()) + n * torch.eye(
        n, dtype=torch.float64, device="cuda")
    del Qs
    A0 = A3.transpose(1, 2).contiguous().view(-1).to(dtype)     # column-major blocks
    del A3, g
    B0 = torch.empty(count * n, dtype=torch.float64, device="cuda")
    tmv_amd.fill_normal(B0, SEED + 52)
    B0 = B0.to(dtype)
    W = torch.empty(count * n, dtype=torch.float64, device="cuda")
    tmv_amd.fill_normal(W, SEED + 53)
    W = W.to(dtype)
    fwd = []
    for _ in range(reps):
        b.A.copy_(A0); b.B.copy_(B0)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        tmv_amd.getrf_batched(b)
        tmv_amd.getrs_batched(b)
        torch.cuda.synchronize()
        fwd.append(time.perf_counter() - t0)
    Xb = tmv_amd.Batch(ns, nr, dtype=dtype, B=b.B.clone())
    Gb = tmv_amd.Batch(ns, nr, dtype=dtype, B=W)
    gB = tmv_amd.Batch(ns, nr, dtype=dtype)
    gA = tmv_amd.Batch(ns, nr, dtype=dtype)
    bwd = []
    for _ in range(reps + 1):
        e0 = torch.cuda.Event(enable_timing=True); e1 = torch.cuda.Event(enable_timing=True)
        e0.record()
        tmv_amd.gesv_adjoint_batched(b, Xb, Gb, gB, gA)
        e1.record()
        torch.cuda.synchronize()
        bwd.append(e0.elapsed_time(e1))
    orig = tmv_amd.Batch(ns, nr, dtype=dtype, A=A0)
    rec = []
    for _ in range(reps):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        tmv_amd.gesv_adjoint_batched(orig, Xb, Gb, gB, gA, recompute=True)
        torch.cuda.synchronize()
        rec.append(time.perf_counter() - t0)
    ms = min(bwd[1:])
    esz = b.A.element_size()
    bytes_ = float(count * (2 * n * n * esz + 3 * n * esz + n * 8))   # LU + gradA, vectors, piv
    return {"systems": count, "n": n, "dtype": str(dtype).replace("torch.", ""),
            "forward_ms": round(min(fwd) * 1e3, 2), "adjoint_ms": round(ms, 3),
            "adjoint_gbs": round(bytes_ / ms / 1e6, 1),
            "adjoint_hbm_frac": round(bytes_ / ms / 1e6 / 8000.0, 4),
            "adjoint_recompute_ms": round(min(rec) * 1e3, 2)}


def _timed(torch, fn, reps=1):
    """Best wall time of fn() over reps runs, device synchronised around each."""
    best = None
    for _ in range(reps):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        fn()
        torch.cuda.synchronize()
        dt = time.perf_counter() - t0
        best = dt if best is None else min(best, dt)
    return best


def _event_ms(torch, fn, reps):
    """Average HIP-event time of fn() on the current stream over reps runs."""
    fn()
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        fn()
    e1.record()
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / reps


def panel_roofline(torch, tmv_amd, A, b, n):
    """The step's dominant kernel, the FP32 panel factorisation: one more
    mixed solve with HIP events around every panel launch (on the stream
    the panel runs on).  Algorithmic bytes: each m x jb FP32 panel read once
    and written once, 8 m jb bytes."""
    tmv_amd.panel_timer_start(4096)
    try:
        tmv_amd.gesv_mixed(A, b, tol=1e-12, max_iter=50)
        torch.cuda.synchronize()
    finally:
        launches, total_ms = tmv_amd.panel_timer_stop()
    nb = next((w for w in (128, 64) if -(-n // w) == launches), 64)   # panel width
    bytes_ = sum(8.0 * (n - j0) * min(nb, n - j0) for j0 in range(0, n, nb))
    per_launch = bytes_ / launches
    avg_ms = total_ms / launches
    achieved = per_launch / (avg_ms * 1e-3) / 1e9
    return {"bound": "hbm", "achieved": round(achieved, 2), "peak": PEAK_HBM_GBS,
            "unit": "GB/s", "frac": round(achieved / PEAK_HBM_GBS, 6),
            "traffic": PANEL_F32_16384_TRAFFIC.get(nb) if n == 16384 else None,
            "kernel": f"panel_kernel<float,{nb},8,512> (FP32 panel of the n={n} mixed solve)",
            "launches": launches, "avg_us": round(avg_ms * 1e3, 2),
            "total_ms": round(total_ms, 3), "bytes_per_launch": round(per_launch),
            "share_of_step": None}


def fp64_lu_solve(torch, tmv_amd, A, b, reps, parts=False):
    """Plain FP64 GPU LU solve (getrf + getrs) on a copy of A: best wall time
    (with parts: also the getrf and getrs times of that run)."""
    best, be, split = None, None, None
    for _ in range(reps):
        LU = A.clone()
        x = b.clone()
        torch.cuda.synchronize()
        t1 = time.perf_counter()
        piv, _ = tmv_amd.getrf(LU)
        torch.cuda.synchronize()
        t2 = time.perf_counter()
        tmv_amd.getrs(LU, piv, x)
        torch.cuda.synchronize()
        t3 = time.perf_counter()
        if best is None or t3 - t1 < best:
            best, split = t3 - t1, (t2 - t1, t3 - t2)
        be = backward_error_gpu(A, x, b, torch)
        del LU, x
    return (best, be, split) if parts else (best, be)


def mixed_section(torch, tmv_amd, a):
    n, nrhs = a.n, a.nrhs
    t_setup = time.perf_counter()
    A = conditioned_gpu(n, a.kappa, SEED + 10, torch, tmv_amd)
    b = torch.empty(n * nrhs, dtype=torch.float64, device="cuda")
    tmv_amd.fill_normal(b, SEED + 12)
    b = b.view(nrhs, n).t() if nrhs > 1 else b
    torch.cuda.synchronize()
    setup_s = time.perf_counter() - t_setup

    # ---- the timed steps: mixed-precision solve ----------------------------
    X = None
    for _ in range(a.warmup):
        X, info = tmv_amd.gesv_mixed(A, b, tol=1e-12, max_iter=50)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    infos = []
    for _ in range(a.steps):
        X, info = tmv_amd.gesv_mixed(A, b, tol=1e-12, max_iter=50)
        infos.append(info)
    torch.cuda.synchronize()
    t_mixed = (time.perf_counter() - t0) / a.steps
    flops = 2.0 / 3.0 * n ** 3 + 2.0 * n * n * nrhs
    be_mixed = backward_error_gpu(A, X, b, torch)
    del X

    roof = panel_roofline(torch, tmv_amd, A, b, n)
    roof["share_of_step"] = round(roof["total_ms"] / (t_mixed * 1e3), 3)

    t_fp64, be64 = fp64_lu_solve(torch, tmv_amd, A, b, a.fp64_reps)
    out = {"value": flops / t_mixed / 1e12, "t_mixed": t_mixed, "setup_s": setup_s,
           "mixed": {"backward_error": be_mixed, "iterations": infos[-1]["iterations"],
                     "converged": infos[-1]["converged"],
                     "factor_ms": round(infos[-1]["factor_ms"], 3),
                     "refine_ms": round(infos[-1]["refine_ms"], 3)},
           "fp64_lu_solve": {"ms": round(t_fp64 * 1e3, 3),
                             "tflops": round(flops / t_fp64 / 1e12, 3),
                             "backward_error": be64},
           "speedup_vs_fp64": round(t_fp64 / t_mixed, 3),
           "roofline_step": roof}

    _progress(f"mixed: {t_mixed * 1e3:.1f} ms/step, panel {roof['avg_us']} us/launch, "
              f"FP64 LU solve {t_fp64 * 1e3:.1f} ms")
    # ---- kappa in {1e2, 1e4, 1e6}: FP32 (1 and 64 RHS), FP16, BF16 -------
    if a.grid:
        grid = {}
        b64 = torch.empty(n * 64, dtype=torch.float64, device="cuda")
        tmv_amd.fill_normal(b64, SEED + 16)
        b64 = b64.view(64, n).t()                 # column-major n x 64
        b1 = b if nrhs == 1 else b[:, 0].contiguous()
        legs = [("f32", tmv_amd.LOWPREC_F32, 1), ("f32", tmv_amd.LOWPREC_F32, 64),
                ("f16", tmv_amd.LOWPREC_F16, 1), ("bf16", tmv_amd.LOWPREC_BF16, 1),
                ("f16x2", tmv_amd.LOWPREC_F16X2, 1), ("bf16x2", tmv_amd.LOWPREC_BF16X2, 1)]
        classic = (tmv_amd.LOWPREC_F32, tmv_amd.LOWPREC_F16X2)   # default refinement
        for kappa, seed in ((1e2, SEED + 14), (a.kappa, None), (1e6, SEED + 18)):
            M = A if seed is None else conditioned_gpu(n, kappa, seed, torch, tmv_amd)
            for name, lp, nr in legs:
                rhs = b1 if nr == 1 else b64
                it = 50 if lp in classic else a.lowp_iter
                tmv_amd.gesv_mixed(M, rhs, tol=1e-12, max_iter=it, lowprec=lp, check=False)
                torch.cuda.synchronize()
                t1 = time.perf_counter()
                Xg, inf = tmv_amd.gesv_mixed(M, rhs, tol=1e-12, max_iter=it, lowprec=lp,
                                             check=False)
                torch.cuda.synchronize()
                dt = time.perf_counter() - t1
                fl = 2.0 / 3.0 * n ** 3 + 2.0 * n * n * nr
                grid[f"kappa{kappa:.0e}_{name}_nrhs{nr}"] = {
                    "ms": round(dt * 1e3, 3), "tflops": round(fl / dt / 1e12, 3),
                    "refine": "classic" if lp in classic else "gmres",
                    "iterations": inf["iterations"], "inner_iterations": inf["inner_iterations"],
                    "converged": inf["converged"], "status": inf["status"],
                    "factor_ms": round(inf["factor_ms"], 3),
                    "refine_ms": round(inf["refine_ms"], 3),
                    "backward_error": backward_error_gpu(M, Xg, rhs, torch)}
                del Xg
                _progress(f"kappa {kappa:.0e} {name} nrhs {nr}: {dt * 1e3:.1f} ms, "
                          f"converged {inf['converged']}")
            for nr, rhs in ((1, b1), (64, b64)):
                t64, be = fp64_lu_solve(torch, tmv_amd, M, rhs, 1)
                grid[f"kappa{kappa:.0e}_fp64_nrhs{nr}"] = {"ms": round(t64 * 1e3, 3),
                                                          "backward_error": be}
            del M
            torch.cuda.empty_cache()
        out["mixed_grid"] = grid
        del b64
    del A
    torch.cuda.empty_cache()
    return out


def fp64_section(torch, tmv_amd, a):
    """DGEMM 8192^3 (CCC, CRC, RCC) and the LU n = 8192 with 16 right-hand
    sides; DGEMM 512^3 and the LU solve n = 512; complex GEMM."""
    out = {}
    gn = a.gemm_n
    GA = torch.empty(gn * gn, dtype=torch.float64, device="cuda")
    GB = torch.empty(gn * gn, dtype=torch.float64, device="cuda")
    tmv_amd.fill_uniform(GA, SEED + 20)
    tmv_amd.fill_uniform(GB, SEED + 21)
    GC = tmv_amd.empty_colmajor(gn, gn, torch.float64)
    gemm = {}
    for lay in ("CC", "CR", "RC"):
        Av = GA.view(gn, gn).t() if lay[0] == "C" else GA.view(gn, gn)
        Bv = GB.view(gn, gn).t() if lay[1] == "C" else GB.view(gn, gn)
        ms = _event_ms(torch, lambda: tmv_amd.gemm(Av, Bv, GC), a.gemm_reps)
        tf = 2.0 * gn ** 3 / ms / 1e9
        name = {"CC": "CCC", "CR": "CRC", "RC": "RCC"}[lay]
        gemm[name] = {"ms": round(ms, 3), "tflops": round(tf, 2),
                      "frac_peak": round(tf / PEAK_FP64_TFLOPS, 4)}
    out["dgemm_8192"] = gemm
    _progress(f"dgemm 8192: {gemm}")
    del GB, GC
    torch.cuda.empty_cache()

    # LU n = 8192, 16 right-hand sides: A uniform[-1,1] (no shift), b ~ N(0,1)
    n = 8192
    A = GA.view(n, n).t() if gn == n else None
    if A is None:
        A = torch.empty(n * n, dtype=torch.float64, device="cuda")
        tmv_amd.fill_uniform(A, SEED + 20)
        A = A.view(n, n).t()
    B16 = torch.empty(n * 16, dtype=torch.float64, device="cuda")
    tmv_amd.fill_normal(B16, SEED + 24)
    B16 = B16.view(16, n).t()
    t, be, (tf, ts) = fp64_lu_solve(torch, tmv_amd, A, B16, 2, parts=True)
    out["lu_8192_nrhs16"] = {"ms": round(t * 1e3, 3),
                             "tflops": round((2 / 3 * n ** 3 + 2 * n * n * 16) / t / 1e12, 3),
                             "getrf_ms": round(tf * 1e3, 3), "getrs_ms": round(ts * 1e3, 3),
                             "backward_error": be}
    del A, GA, B16
    torch.cuda.empty_cache()

    # the CPU-sized case: DGEMM 512^3, LU solve n = 512 (A + n I, 1 RHS)
    n = 512
    A = torch.empty(n * n, dtype=torch.float64, device="cuda")
    B = torch.empty(n * n, dtype=torch.float64, device="cuda")
    tmv_amd.fill_uniform(A, SEED + 100)
    tmv_amd.fill_uniform(B, SEED + 101)
    Av, Bv = A.view(n, n).t(), B.view(n, n).t()
    C = tmv_amd.empty_colmajor(n, n, torch.float64)
    g_us = _event_ms(torch, lambda: tmv_amd.gemm(Av, Bv, C), 200) * 1e3
    g_wall = _timed(torch, lambda: tmv_amd.gemm(Av, Bv, C), 20) * 1e6
    M = Av.clone()
    M.diagonal().add_(float(n))
    bb = torch.empty(n, dtype=torch.float64, device="cuda")
    tmv_amd.fill_uniform(bb, SEED + 102)
    t, be, (tf, ts) = fp64_lu_solve(torch, tmv_amd, M, bb, 20, parts=True)
    out["cfg512"] = {"dgemm_us": round(g_us, 2), "dgemm_wall_us": round(g_wall, 2),
                     "dgemm_tflops": round(2 * n ** 3 / g_us / 1e6, 3),
                     "lu_solve_us": round(t * 1e6, 1), "getrf_us": round(tf * 1e6, 1),
                     "getrs_us": round(ts * 1e6, 1),
                     "lu_solve_gflops": round((2 / 3 * n ** 3 + 2 * n * n) / t / 1e9, 2),
                     "lu_backward_error": be}
    del A, B, C, M
    torch.cuda.empty_cache()

    # ---- complex GEMM (TMV's four-real-product split), complex128 CCC ------
    zn = a.zgemm_n
    if zn > 0:
        ZA = torch.empty(2 * zn * zn, dtype=torch.float64, device="cuda")
        ZB = torch.empty(2 * zn * zn, dtype=torch.float64, device="cuda")
        tmv_amd.fill_uniform(ZA, SEED + 22)
        tmv_amd.fill_uniform(ZB, SEED + 23)
        ZAv = torch.view_as_complex(ZA.view(zn, zn, 2)).t()
        ZBv = torch.view_as_complex(ZB.view(zn, zn, 2)).t()
        ZC = tmv_amd.empty_colmajor(zn, zn, torch.complex128)
        ms = _event_ms(torch, lambda: tmv_amd.gemm_complex(ZAv, ZBv, ZC), a.gemm_reps)
        tf = 8.0 * zn ** 3 / ms / 1e9
        out["zgemm"] = {"n": zn, "ms": round(ms, 3), "tflops": round(tf, 2),
                        "frac_peak": round(tf / PEAK_FP64_TFLOPS, 4),
                        "flops": "8 n^3 real (4 real products)"}
        del ZA, ZB, ZC, ZAv, ZBv
        torch.cuda.empty_cache()
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=5)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--n", type=int, default=16384)
    ap.add_argument("--kappa", type=float, default=1e4)
    ap.add_argument("--nrhs", type=int, default=1)
    ap.add_argument("--fp64-reps", type=int, default=2)
    ap.add_argument("--lowp-iter", type=int, default=4,
                    help="outer refinement steps for the FP16/BF16 legs (GMRES-IR)")
    ap.add_argument("--gemm-n", type=int, default=8192)
    ap.add_argument("--gemm-reps", type=int, default=5)
    ap.add_argument("--zgemm-n", type=int, default=8192, help="complex GEMM size (0: skip)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--cpu-cfg2", action="store_true",
                    help="also time TMV on the 8192 case (minutes of CPU)")
    ap.add_argument("--cpu-reps", type=int, default=3)
    ap.add_argument("--no-batched", action="store_true")
    ap.add_argument("--no-grid", dest="grid", action="store_false",
                    help="skip the kappa grid of mixed solves")
    ap.add_argument("--only", choices=["mixed", "fp64", "batched", "cpu"], default=None)
    ap.add_argument("--only-batched", action="store_true", help="same as --only batched")
    a = ap.parse_args()
    if a.gpus != 1:
        print(f"bench.py runs on one GPU only (asked for --gpus {a.gpus}): every figure is "
              "one GPU's; the multi-GPU layout is a design, not measured", file=sys.stderr)
        sys.exit(2)
    if a.only_batched:
        a.only = "batched"

    if a.only == "cpu":                 # TMV on the host alone (no GPU)
        print(json.dumps({"cpu_baseline": cpu_baseline(),
                          "cpu_configs": cpu_configs(a.cpu_cfg2, a.cpu_reps)}), flush=True)
        return

    import torch
    import tmv_amd
    tmv_amd.lib()                      # the HIP library; no fallback
    if a.only == "batched":            # the batched workloads alone (profiling)
        print(json.dumps({"batched_20000": {
            "f64": batched_workload(torch, tmv_amd, torch.float64),
            "f32": batched_workload(torch, tmv_amd, torch.float32)},
            "adjoint_512x256": {
            "f64": adjoint_workload(torch, tmv_amd, torch.float64),
            "f32": adjoint_workload(torch, tmv_amd, torch.float32)}}), flush=True)
        return
    if a.only == "fp64":
        print(json.dumps(fp64_section(torch, tmv_amd, a)), flush=True)
        return

    mx = mixed_section(torch, tmv_amd, a)
    if a.only == "mixed":
        mx.pop("t_mixed")
        print(json.dumps(mx), flush=True)
        return
    f64 = fp64_section(torch, tmv_amd, a)
    _progress("fp64 section done")

    batched = adjoint = None
    if not a.no_batched:
        batched = {"f64": batched_workload(torch, tmv_amd, torch.float64),
                   "f32": batched_workload(torch, tmv_amd, torch.float32)}
        adjoint = {"f64": adjoint_workload(torch, tmv_amd, torch.float64),
                   "f32": adjoint_workload(torch, tmv_amd, torch.float32)}

    _progress("GPU sections done")
    cpu = cpu_cfg = None
    if not a.no_cpu_baseline:
        try:
            cpu = cpu_baseline()
        except Exception as ex:          # reported, never silently replaced
            cpu = {"value": None, "unit": "TFLOP/s", "cores": None, "kind": "reference",
                   "sample": f"failed: {ex}"}
        try:
            cpu_cfg = cpu_configs(a.cpu_cfg2, a.cpu_reps)
        except Exception as ex:
            cpu_cfg = {"failed": str(ex)}

    ccc = f64["dgemm_8192"]["CCC"]
    gn = a.gemm_n
    out = {
        "metric": "LU-solve TFLOP/s: FP32-MFMA+IR vs FP64 at <=1e-12 backward err; DGEMM % peak",
        "value": round(mx["value"], 3),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": a.steps,
        "warmup": a.warmup,
        "ms_per_step": round(mx["t_mixed"] * 1e3, 3),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32 factorisation + f64 refinement",
        "data": "synthetic: A = U diag(s) V^T (QR of seeded Gaussians), b ~ N(0,1)",
        "config": {"workload": "mixed-precision LU solve + iterative refinement",
                   "n": a.n, "nrhs": a.nrhs, "kappa": a.kappa, "target_backward_error": 1e-12,
                   "parallelism": "single GPU"},
        "mixed": mx["mixed"],
        "fp64_lu_solve": mx["fp64_lu_solve"],
        "speedup_vs_fp64": mx["speedup_vs_fp64"],
        "mixed_grid": mx.get("mixed_grid"),
        "dgemm_8192": f64["dgemm_8192"],
        "lu_8192_nrhs16": f64["lu_8192_nrhs16"],
        "cfg512": f64["cfg512"],
        "zgemm": f64.get("zgemm"),
        "batched_20000": batched,
        "adjoint_512x256": adjoint,
        "roofline": {"bound": "mfma", "achieved": ccc["tflops"], "peak": PEAK_FP64_TFLOPS,
                     "unit": "TFLOP/s", "frac": ccc["frac_peak"],
                     "traffic": DGEMM_8192_CCC_TRAFFIC if gn == 8192 else None,
                     "kernel": "gemm_kernel f64 128x128x16 (DGEMM 8192^3, CCC)",
                     "flops_per_launch": 2 * gn ** 3},
        "roofline_step": mx["roofline_step"],
        "cpu_baseline": cpu,
        "cpu_configs": cpu_cfg,
        "setup_s": round(mx["setup_s"], 1),
    }
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
