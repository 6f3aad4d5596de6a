"""Benchmark: wall time of exp(-iHt)psi at 1e-6 error for sparse SYK N=48,
plus the HBM bandwidth the Pauli apply sustains.

Workload (one "step"): sparse SYK q=4, N=48 Majoranas (24 qubits, dim 2^24),
k=8 (Bernoulli-kept quadruples, ~kN=384 terms), generated by the C++ API's
SYK::gen_ham with std::mt19937(seed); a seeded complex Gaussian initial
state; restarted Krylov to t=10 with FP32 state vectors, FP64 reductions and
an FP64 Hessenberg exponential, the Krylov dimension of each restart proposed
by the trained proposer network (reapers_amd/proposer.f32, evaluated by the
HIP inference kernel; a rejected proposal falls back to dimension 20).  The error of the FP32
result is measured against an FP64 evolution of the same (promoted)
Hamiltonian and state at a tight tolerance, outside the timed region.

Reported beside it: the plain FP64 single-state Krylov (fixed dimension 20)
and the FP32 evolution with the fixed dimension 20 on the same GPU; four
states sharing the Hamiltonian evolved as one batch (seconds per state); the
apply kernel's roofline (HBM-side bytes per launch from rocprofv3 counters
under profiles/, over the kernel's average duration from HIP events on the
library stream, with the tile-stream bytes and on-chip rates beside it), for
the headline's 24 qubits and for a 30-qubit apply whose state leaves every
cache; and the reference's CPU algorithm (the oracle, production flags)
timed on bounded samples.

python bench.py [--steps K] [--warmup W] [--gpus 1]
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "exp(-iHt)ψ wall time at 1e-6 err (sparse SYK N=48) + Pauli-apply HBM GB/s"
HBM_PEAK_GBS = 8000.0


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def traffic_record(name, tiling, kernel=None):
    """The counter-measured bytes per launch of the apply kernel for one
    tiling (tile bits, threads, depth): rocprofv3 FETCH_SIZE and WRITE_SIZE
    passes, each scaled by what the counter reads for a streaming kernel of
    known size, recorded under profiles/; None when that tiling (and, given
    `kernel`, that kernel) was not measured."""
    p = os.path.join(ROOT, "profiles", name)
    if not os.path.exists(p):
        return None
    try:
        with open(p) as f:
            d = json.load(f)
    except Exception:
        return None
    if list(d.get("tiling", [])) != list(tiling):
        return None
    if kernel is not None and d.get("kernel") != kernel:
        return None
    return d


# on-chip peaks of one MI355X used beside the HBM roofline: 256 CUs at
# 2.4 GHz; LDS 128 bytes per clock per CU; non-packed FP32 FMA 64 lanes per
# clock per CU (packed FP32 is not used by this build)
N_CU, CLOCK_GHZ = 256, 2.4
LDS_PEAK_TBS = N_CU * 128 * CLOCK_GHZ / 1e3
FP32_VALU_TFLOPS = N_CU * 64 * 2 * CLOCK_GHZ / 1e3


def apply_kernel_name(info):
    """The apply kernel a term handle launches, as rocprofv3 names it (the
    template arguments shortened)."""
    import reapers_amd as ra
    if info.kernel == ra.RP_APPLY_STREAM:
        return "k_apply_stream<b=%d,threads=%d>" % (info.tile_bits, info.threads)
    if info.kernel == ra.RP_APPLY_SMALL:
        return "k_apply_wave"
    return "k_apply_tiled<%s,b=%d,threads=%d,depth=%d>" % (
        "float" if info.prec == ra.RP_C64 else "double", info.tile_bits, info.threads,
        info.depth)


def apply_roofline(info, avg_ms, L, traffic_name):
    """Roofline object of one apply kernel: achieved = HBM-side bytes per
    launch (counter-measured, profiles/) over the kernel's average launch
    time; beside it the tile-stream bytes (G_b + 1) * 2^L * 8 that the
    L2/Infinity Cache serve, and the LDS and FMA rates of the term loop."""
    secs = avg_ms / 1e3
    rec = traffic_record(traffic_name, (info.tile_bits, info.threads, info.depth),
                         apply_kernel_name(info))
    traffic = None if rec is None else int(rec["hbm_bytes_per_launch"])
    achieved = None if traffic is None else traffic / secs / 1e9
    term_apps = info.nterms * (1 << L)
    obj = {
        "bound": "hbm",
        "achieved": None if achieved is None else round(achieved, 1),
        "peak": HBM_PEAK_GBS,
        "unit": "GB/s",
        "frac": None if achieved is None else round(achieved / HBM_PEAK_GBS, 4),
        "traffic": traffic,
        "traffic_source": None if rec is None else "profiles/%s (%s)" % (traffic_name,
                                                                        rec.get("source", "")),
        "kernel": apply_kernel_name(info),
        "avg_launch_ms": round(avg_ms, 4),
        "tile_stream": {
            "model": "(G_b+1) * 2^L * 8 B: each input tile staged once per tile group, "
                     "plus the output write; served by L2 and the Infinity Cache",
            "bytes_per_launch": int(info.bytes_per_apply), "groups_G_b": int(info.ngroups),
            "TBps": round(info.bytes_per_apply / secs / 1e12, 2)},
        "onchip": {
            "term_apps_per_s": float("%.4g" % (term_apps / secs)),
            "lds_read_TBps": round(term_apps * 8 / secs / 1e12, 2),
            "lds_peak_TBps": round(LDS_PEAK_TBS, 1),
            "fma_TFLOPs": round(term_apps * 4 / secs / 1e12, 2),
            "fp32_valu_peak_TFLOPs": round(FP32_VALU_TFLOPS, 1),
            "note": "one 8-byte LDS read and two FP32 FMAs per term application"},
    }
    return obj


def n60_apply(ra, otoc_point=False):
    """The apply at 30 qubits (sparse SYK N=60, the OTOC workload's 8.6 GB
    complex<float> state, which no cache holds): uploaded as the OTOC mode
    uploads it (tiling autotuner, group accumulation), then one warm-up and
    three launches of the kept tiling, HIP events on the library stream; the
    roofline from the counter-measured bytes of that tiling."""
    import ctypes
    N, L = 60, 30
    hip = ra.hip()
    bits, coeff = ra.syk_terms(N, 8.0, seed=4000, fp=32)
    H = ra.Hamiltonian(L, bits, coeff, fp=32)
    info = H.info()          # the device upload (and the tiling trials) happen here
    a = ra.DeviceState(L, fp=32)
    a.random(4001)
    b = ra.DeviceState(L, fp=32)
    b.copy_from(a)
    b.apply(H)
    ra.check(hip.rp_synchronize())
    ra.check(hip.rp_prof_reset())
    ra.check(hip.rp_prof_enable(0x100 | (1 << ra.RP_KERNEL_APPLY)))
    for _ in range(3):
        b.copy_from(a)
        b.apply(H)
    ra.check(hip.rp_synchronize())
    n, ms = ctypes.c_uint64(), ctypes.c_double()
    ra.check(hip.rp_prof_query(ra.RP_KERNEL_APPLY, ctypes.byref(n), ctypes.byref(ms)))
    ra.check(hip.rp_prof_enable(0))
    avg = ms.value / max(n.value, 1)
    log("N=60 apply: %d terms, %d groups, %.2f ms per launch" % (info.nterms, info.ngroups, avg))
    obj = apply_roofline(info, avg, L, "apply_c64_syk60_traffic.json")
    obj["workload"] = "sparse SYK k=8 N=60, 30 qubits, %d terms, complex<float> (8.6 GB state)" % (
        info.nterms)
    obj["launches"] = int(n.value)
    b.close()
    otoc = None
    if otoc_point:
        try:
            otoc = otoc_first_point(ra, H, a, N, L)
        except Exception as e:      # recorded, not fatal to the headline line
            otoc = {"error": "%s: %s" % (type(e).__name__, e)}
    a.close()
    H.close()
    return obj, otoc


def otoc_first_point(ra, H, s, N, L):
    """Configuration 4's first time point: the OTOC of sparse SYK N=60 at
    t = 0.1 (the first of the 20 log-spaced times in [0.1, 20]), W = chi_1,
    V = chi_2, beta = 0, Krylov dimensions from the trained proposer
    (fallback 12, capped by what fits in HBM), on the Hamiltonian the apply
    line uploaded."""
    import ctypes
    from reapers_amd import proposer
    hip = ra.hip()
    ops = []
    for idx in (1, 2):
        mb, mc = ra.majorana(N, idx, fp=32)
        ops.append(ra.Hamiltonian(L, np.array([mb], np.uint64), np.array([mc]), fp=32))
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    ra.check(hip.rp_mem_get_info(ctypes.byref(free), ctypes.byref(total)))
    max_dim = int(max(12, min(40, free.value // (8 << L) - 4)))
    sched = ra.Schedule.from_mlp(proposer.load_weights(), max_dim=max_dim)
    tk = float(np.geomspace(0.1, 20.0, 20)[0])
    s.random(4001)
    ra.check(hip.rp_synchronize())
    t0 = time.perf_counter()
    F, st = s.otoc(H, ops[0], ops[1], [tk], krydim=12, tol=1e-7, schedule=sched)
    wall = time.perf_counter() - t0
    sched.close()
    for o in ops:
        o.close()
    log("N=60 OTOC t=%.4g: F=%.8g%+.3gi, %.2fs, %d matvecs" % (tk, F[0].real, F[0].imag, wall,
                                                              st.matvecs))
    return {"t": tk, "F": [float("%.8g" % F[0].real), float("%.8g" % F[0].imag)],
            "s_per_point": round(wall, 3), "matvecs": int(st.matvecs),
            "rejected_proposals": int(st.rejected), "proposer_max_dim": max_dim,
            "workload": "sparse SYK k=8 N=60 (30 qubits), W=chi_1, V=chi_2, beta=0, first of the "
                        "20 log-spaced times, proposer-chosen Krylov dims (fallback 12), FP32 "
                        "states, FP64 reductions, tol 1e-7"}


def cpu_baseline(bits, coeff, L, psi, matvecs, target_s):
    """The reference's CPU algorithm (the oracle's restatement of
    CPUImpl::apply_ops, inc/cpuimpl.h:737-754, and Krylov::evolve,
    inc/algo.h:266-365) built with the production flags (liboracle_fast.so:
    -O3, AVX2/FMA, OpenMP on every host core), timed on bounded samples: the
    N=48 apply on a row sample, one apply at N=24..40, and the whole FP32
    evolution (t=10, tol 1e-7, dimension 20) at N=32 and N=36.  value = the
    N=48 evolution extrapolated from the N=36 one: its time per matvec
    (apply, Gram-Schmidt and Hessenberg work together) scaled by the ratio of
    the N=48 and N=36 apply times, times the GPU run's matvec count."""
    import oracle
    import time as _t
    with oracle.use(oracle.fast()):
        dim = 1 << L
        rows = 1 << 12
        oracle.apply_rows_timed(L, bits, coeff, psi, rows, fp=32)
        t, _ = oracle.apply_rows_timed(L, bits, coeff, psi, rows, fp=32)
        rows = int(min(dim, max(rows, rows * target_s / max(t, 1e-6))))
        t, _ = oracle.apply_rows_timed(L, bits, coeff, psi, rows, fp=32)
        apply48 = t * dim / rows
        per_apply = {"48": round(apply48, 3)}
        evo = {}
        rng = np.random.default_rng(36)
        for N in (24, 32, 36, 40):
            Ls = N // 2
            b, c = oracle.syk_terms(N, 8.0, seed=2000 + N, fp=32)
            p = (rng.standard_normal(1 << Ls) + 1j * rng.standard_normal(1 << Ls))
            p = (p / np.linalg.norm(p)).astype(np.complex64)
            oracle.apply_rows_timed(Ls, b, c, p, 1 << Ls, fp=32)
            ta, _ = oracle.apply_rows_timed(Ls, b, c, p, 1 << Ls, fp=32)
            per_apply[str(N)] = round(ta, 4)
            if N in (32, 36):
                t0 = _t.perf_counter()
                _, st = oracle.krylov_evolve(Ls, b, c, p, 10.0, 0.0, krydim=20, tol=1e-7, fp=32)
                tt = _t.perf_counter() - t0
                evo[str(N)] = {"s": round(tt, 3), "matvecs": int(st.matvecs),
                               "s_per_matvec": round(tt / max(st.matvecs, 1), 4)}
        per_mv36 = evo["36"]["s_per_matvec"]
        value = per_mv36 * (apply48 / per_apply["36"]) * matvecs
    return {
        "value": round(value, 2),
        "unit": "s",
        "cores": oracle.num_threads(),
        "kind": "port",
        "sample": ("extrapolated N=48 evolution: the whole N=36 evolution's %.3f s per matvec x "
                   "the N=48/N=36 apply-time ratio %.1f (N=48 apply %.2f s from rows [0,%d), "
                   "%.1f%% of the state) x %d matvecs; oracle built -O3 -march=x86-64-v3 "
                   "-fopenmp" % (per_mv36, apply48 / per_apply["36"], apply48, rows,
                                 100.0 * rows / dim, matvecs)),
        "apply_s": per_apply,
        "evolution_t10_tol1e-7_dim20": evo,
        "cpu_model": _cpu_model(),
    }


def _cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except Exception:
        pass
    return None


def apply_only(ra, args, bits, coeff, L, psi0):
    """Time K applies of H (one state precision after the other) with HIP
    events on the library stream; one JSON line per precision."""
    import ctypes
    hip = ra.hip()
    fps = (32, 64) if args.apply_fp == "both" else (int(args.apply_fp),)
    for fp in fps:
        H = ra.Hamiltonian(L, bits, coeff, fp=fp)
        info = H.info()
        s = ra.DeviceState(L, fp=fp)
        s.copy_from(psi0)
        for _ in range(args.warmup):
            s.apply(H)
        ra.check(hip.rp_prof_reset())
        ra.check(hip.rp_prof_enable(1))
        t0 = time.perf_counter()
        for _ in range(args.steps):
            s.apply(H)
        ra.check(hip.rp_synchronize())
        wall = time.perf_counter() - t0
        n, ms = ctypes.c_uint64(), ctypes.c_double()
        ra.check(hip.rp_prof_query(ra.RP_KERNEL_APPLY, ctypes.byref(n), ctypes.byref(ms)))
        ra.check(hip.rp_prof_enable(0))
        avg = ms.value / max(n.value, 1)
        print(json.dumps({
            "mode": "apply", "fp": fp, "launches": n.value, "avg_launch_ms": round(avg, 4),
            "wall_ms_per_apply": round(wall * 1e3 / args.steps, 4),
            "tile_bits": info.tile_bits, "groups": int(info.ngroups), "terms": int(info.nterms),
            "tile_stream_bytes_per_launch": int(info.bytes_per_apply),
            "tile_stream_GBps": round(info.bytes_per_apply / (avg / 1e3) / 1e9, 1),
            "term_apps_per_s": float("%.4g" % (info.nterms * (1 << L) / (avg / 1e3))),
        }), flush=True)
        s.close()
        H.close()
    # calibration for hardware byte counters: one complex<float> ->
    # complex<double> conversion of the state, which reads 8 and writes 16
    # bytes per amplitude (kernel k_f2d)
    d = ra.DeviceState(L, fp=64)
    d.copy_from(psi0)
    ra.check(hip.rp_synchronize())
    print(json.dumps({"mode": "calibration", "kernel": "k_f2d", "read_bytes": 8 << L,
                      "write_bytes": 16 << L}), flush=True)
    d.close()


def batch_mode(ra, args):
    print(json.dumps(batch_result(ra, single=True)), flush=True)


def batch_result(ra, single=True):
    """64 sparse SYK k=8 realizations (seed 3000 + r) of N drawn from
    {32, 36, 40, 44}, 4 seeded random states each: 256 right-hand sides
    evolved to t=5 at tol 1e-6 in one batch (FP32 states, FP64 reductions,
    graph-replayed restarts, autotuned apply tiling), against the same 256
    evolutions one state at a time through the single-state path (single;
    otherwise only the error sample's 16 states are evolved alone, in FP64)."""
    nreal, nrhs, t, tol, m, kmax = 64, 4, 5.0, 1e-6, 12, 24
    rng = np.random.default_rng(3)
    Ns = rng.choice([32, 36, 40, 44], size=nreal)
    lens = [int(n) // 2 for n in Ns]
    terms = [ra.syk_terms(int(n), 8.0, seed=3000 + r, fp=32) for r, n in enumerate(Ns)]
    states = []
    for L in lens:
        x = rng.normal(size=(1 << L, nrhs)) + 1j * rng.normal(size=(1 << L, nrhs))
        states.append((x / np.linalg.norm(x, axis=0)).astype(np.complex64))
    t0 = time.perf_counter()
    b = ra.Batch(lens, terms, nrhs=nrhs, kmax=kmax, fp=32, autotune=True)
    log("batch: %d problems, %d rhs, %.2f GB per vector, tiling b=%d/%d threads, grid %d "
        "(built and tuned in %.1fs)" % (nreal, nreal * nrhs, b.info.vec_bytes / 1e9,
                                         b.info.tile_bits, b.info.threads, b.info.grid,
                                         time.perf_counter() - t0))
    b.load(states)
    b.evolve(t, m=m, tol=tol)            # warm-up
    b.load(states)
    ra.check(ra.hip().rp_synchronize())
    t0 = time.perf_counter()
    st, rs = b.evolve(t, m=m, tol=tol)
    batch_s = time.perf_counter() - t0
    got = b.store()
    # the same batch with the proposer choosing each restart's dimension
    from reapers_amd import proposer
    sched = ra.Schedule.from_mlp(proposer.load_weights(), max_dim=kmax)
    b.load(states)
    b.evolve(t, m=m, tol=tol, schedule=sched)    # warm-up (captures the graphs)
    b.load(states)
    ra.check(ra.hip().rp_synchronize())
    t0 = time.perf_counter()
    st_p, rs_p = b.evolve(t, m=m, tol=tol, schedule=sched)
    batch_p_s = time.perf_counter() - t0
    got_p = b.store()
    # batched apply timing (HIP events) for the roofline
    import ctypes
    hip = ra.hip()
    ra.check(hip.rp_prof_reset())
    ra.check(hip.rp_prof_enable(1))
    for _ in range(3):
        b.apply()
    ra.check(hip.rp_synchronize())
    n, ms = ctypes.c_uint64(), ctypes.c_double()
    ra.check(hip.rp_prof_query(ra.RP_KERNEL_APPLY, ctypes.byref(n), ctypes.byref(ms)))
    ra.check(hip.rp_prof_enable(0))
    apply_ms = ms.value / max(n.value, 1)
    bpl = int(b.info.bytes_per_apply)
    b.close()
    # the same 256 evolutions one state at a time (single-state FP32 path)
    single_s = 0.0
    errs, errs_p = [], []
    for p, L in enumerate(lens):
        check = p < 4
        if not single and not check:
            break
        H = ra.Hamiltonian(L, *terms[p], fp=32)
        s1 = ra.DeviceState(L, fp=32)
        if check:
            H64 = ra.Hamiltonian(L, *terms[p], fp=64)
            s64 = ra.DeviceState(L, fp=64)
        for q in range(nrhs):
            if single:
                s1.load(states[p][:, q])
                ra.check(hip.rp_synchronize())
                t1 = time.perf_counter()
                s1.evolve(H, t, 0.0, krydim=m, tol=tol)
                single_s += time.perf_counter() - t1
            if check:
                s64.load(states[p][:, q].astype(np.complex128))
                s64.evolve(H64, t, 0.0, krydim=30, tol=1e-13)
                ref = s64.store()
                errs.append(float(np.linalg.norm(got[p][:, q] - ref) / np.linalg.norm(ref)))
                errs_p.append(float(np.linalg.norm(got_p[p][:, q] - ref) / np.linalg.norm(ref)))
        s1.close()
        H.close()
        if check:
            s64.close()
            H64.close()
    line = {
        "mode": "batch",
        "metric": "right-hand sides evolved per second (batched sparse SYK)",
        "value": round(nreal * nrhs / batch_s, 2), "unit": "rhs/s",
        "batch_s": round(batch_s, 4), "single_state_s": round(single_s, 4) if single else None,
        "speedup_vs_single_state": round(single_s / batch_s, 3) if single else None,
        "proposer": {"batch_s": round(batch_p_s, 4), "rhs_per_s": round(nreal * nrhs / batch_p_s, 2),
                     "matvecs_rhs": int(st_p.matvecs), "restarts_max": int(rs_p.max()),
                     "rejected": int(st_p.rejected),
                     "max_err_vs_fp64_sample": max(errs_p)},
        "config": {"workload": "64 sparse SYK k=8 realizations, N in {32,36,40,44}, 4 states "
                               "each, exp(-iHt) to t=5, tol 1e-6, Krylov dim 12, FP32",
                   "N_counts": {int(k): int((Ns == k).sum()) for k in (32, 36, 40, 44)}},
        "restarts_max": int(rs.max()), "restarts_min": int(rs.min()),
        "matvecs_rhs": int(st.matvecs), "host_ms": round(st.host_ms, 1),
        "max_err_vs_fp64_sample": max(errs), "err_sample": "16 rhs of the first 4 realizations",
        "apply": {"kernel": "k_batch_apply", "avg_launch_ms": round(apply_ms, 3),
                  "tile_stream_bytes_per_launch": bpl,
                  "tile_stream_GBps": round(bpl / (apply_ms / 1e3) / 1e9, 1)},
    }
    return line


def otoc_mode(ra, args):
    """OTOC of sparse SYK k=8, N=60 (30 qubits, FP32 state 8.6 GB), W = chi_1,
    V = chi_2, Krylov dimensions from the trained proposer (fallback 12;
    also the fixed dimension 12 unless --no-fixed), at the first
    --otoc-points of the 20 log-spaced times in [0.1, 20]; plus the apply's
    roofline at this size."""
    import ctypes
    N, L = 60, 30
    hip = ra.hip()
    t0 = time.perf_counter()
    bits, coeff = ra.syk_terms(N, 8.0, seed=4000, fp=32)
    H = ra.Hamiltonian(L, bits, coeff, fp=32)
    info = H.info()
    log("N=60: %d terms, groups %d, generated in %.1fs" % (info.nterms, info.ngroups,
                                                           time.perf_counter() - t0))
    s = ra.DeviceState(L, fp=32)
    s.random(4001)
    ra.check(hip.rp_prof_reset())
    ra.check(hip.rp_prof_enable(1))
    for _ in range(3):
        s.apply(H)
    ra.check(hip.rp_synchronize())
    n, ms = ctypes.c_uint64(), ctypes.c_double()
    ra.check(hip.rp_prof_query(ra.RP_KERNEL_APPLY, ctypes.byref(n), ctypes.byref(ms)))
    ra.check(hip.rp_prof_enable(0))
    apply_ms = ms.value / max(n.value, 1)
    log("apply: %.2f ms, %.0f GB/s of tile stream" % (apply_ms,
                                                       info.bytes_per_apply / apply_ms / 1e6))
    s.random(4001)
    ops = []
    for idx in (1, 2):
        mb, mc = ra.majorana(N, idx, fp=32)
        ops.append(ra.Hamiltonian(L, np.array([mb], np.uint64), np.array([mc]), fp=32))
    A, B = ops
    times = np.geomspace(0.1, 20.0, 20)[:args.otoc_points]
    from reapers_amd import proposer
    # the proposer's largest dimension is bounded by what fits: the OTOC
    # holds the initial state and one evolving state with m + 2 vectors
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    ra.check(hip.rp_mem_get_info(ctypes.byref(free), ctypes.byref(total)))
    vec_bytes = 8 << L
    max_dim = int(max(12, min(40, free.value // vec_bytes - 4)))
    log("free %.1f GB: proposer dimensions capped at %d" % (free.value / 1e9, max_dim))
    sched = ra.Schedule.from_mlp(proposer.load_weights(), max_dim=max_dim)
    # one call per time point (beta = 0: the points are independent), with a
    # progress line after each
    F = np.zeros(len(times), complex)
    st = ra.EvolveStats()
    per_point = []
    t0 = time.perf_counter()
    for i, tk in enumerate(times):
        tp = time.perf_counter()
        Fi, sti = s.otoc(H, A, B, [tk], krydim=12, tol=1e-7, schedule=sched)
        F[i] = Fi[0]
        st.matvecs += sti.matvecs
        st.restarts += sti.restarts
        st.rejected += sti.rejected
        per_point.append(round(time.perf_counter() - tp, 3))
        log("t=%.4g: F=%.8g%+.3gi, %.2fs, %d matvecs" % (tk, F[i].real, F[i].imag, per_point[-1],
                                                        sti.matvecs))
    wall = time.perf_counter() - t0
    log("OTOC with the proposer: %.2fs, %d matvecs" % (wall, st.matvecs))
    fixed = None
    if len(times) and not args.no_fixed:
        s.random(4001)
        t0 = time.perf_counter()
        Ff, stf = s.otoc(H, A, B, times, krydim=12, tol=1e-7)
        wf = time.perf_counter() - t0
        fixed = {"s_per_point": round(wf / len(times), 3), "matvecs": int(stf.matvecs),
                 "max_abs_diff_F": float(np.abs(Ff - F).max())}
        log("OTOC with Krylov dim 12: %.2fs, %d matvecs" % (wf, stf.matvecs))
    line = {
        "mode": "otoc", "metric": "OTOC wall time per time point (sparse SYK N=60)",
        "value": round(wall / len(times), 3) if len(times) else None, "unit": "s",
        "times": [float("%.4g" % x) for x in times],
        "F": [[float("%.8g" % v.real), float("%.8g" % v.imag)] for v in F],
        "matvecs": int(st.matvecs), "restarts": int(st.restarts),
        "rejected_proposals": int(st.rejected), "proposer_max_dim": max_dim, "fixed_dim_12": fixed,
        "s_per_point": per_point, "total_s": round(wall, 3),
        "config": {"workload": "sparse SYK k=8 N=60 (30 qubits), W=chi_1, V=chi_2, proposer-chosen "
                               "Krylov dims (fallback 12), FP32 states, FP64 reductions",
                   "terms": int(info.nterms)},
        "roofline": apply_roofline(info, apply_ms, L, "apply_c64_syk60_traffic.json"),
    }
    print(json.dumps(line), flush=True)


def proposer_mode(ra, args):
    print(json.dumps(proposer_result(ra)), flush=True)


def proposer_result(ra):
    """The trained Krylov-schedule proposer against the fixed dimension 20 on
    sizes it was not trained on: random-field XXZ chains of 26 sites and
    sparse SYK N=48, FP32 states at tol 1e-7, error against an FP64
    evolution; matvecs and wall time per evolution."""
    from reapers_amd import proposer
    rng = np.random.default_rng(5150)
    insts = [proposer.make_instance(rng, "xxz", 26, fp=32) for _ in range(3)]
    insts += [proposer.make_instance(rng, "syk", 24, fp=32) for _ in range(3)]
    for d, *_ in insts:
        d["tol"] = 1e-7
    rows = proposer.evaluate(proposer.load_weights(), insts, fixed=20, fp=32, log=log)
    keep = ("kind", "L", "t", "W", "Delta", "seed", "matvecs_fixed", "matvecs_mlp", "wall_ms_fixed",
            "wall_ms_mlp", "err_fixed", "err_mlp", "dims_mlp", "nsub_mlp", "rejected_mlp")
    out = [{k: r[k] for k in keep if k in r} for r in rows]
    tot = {k: sum(r[k] for r in rows) for k in ("matvecs_fixed", "matvecs_mlp", "wall_ms_fixed",
                                                 "wall_ms_mlp")}
    return {
        "mode": "proposer", "metric": "matvecs and wall time per exp(-iHt)psi, proposer vs fixed "
                                      "Krylov dimension 20 (unseen XXZ L=26 and SYK N=48)",
        "value": round(tot["wall_ms_fixed"] / tot["wall_ms_mlp"], 3), "unit": "x wall-time speedup",
        "matvecs_speedup": round(tot["matvecs_fixed"] / tot["matvecs_mlp"], 3),
        "max_err_mlp": max(r["err_mlp"] for r in rows), "max_err_fixed": max(r["err_fixed"] for r in rows),
        "totals": tot, "instances": out}


def _prof_query(ra, cls):
    import ctypes
    n, ms = ctypes.c_uint64(), ctypes.c_double()
    ra.check(ra.hip().rp_prof_query(cls, ctypes.byref(n), ctypes.byref(ms)))
    return n.value, ms.value


def block_mode(ra, args):
    """The reference's production path: one disorder realization of the
    parity-block SYK OTOC driver (examples/syk.cc:120-284) for sparse SYK
    k=8, N=48 (two sectors of 23 qubits): Lanczos E0 of H_L, the shift, the
    beta/8 pre-evolution, then per time point t_k = k tmax/nsteps four FP32
    Krylov evolutions (tol 1e-7, Krylov dimensions from the trained proposer,
    fallback 20) and two Majorana applications.  value = wall time per
    nonzero time point, beside the fixed dimension 20; the apply's roofline
    at 2^23."""
    N, k, seed, beta, tmax = 48, 8.0, args.seed, 1.0, 10.0
    L = N // 2 - 1
    bL, cL = ra.syk_block_terms(N, 0, k, seed=seed, fp=32)
    info = ra.Hamiltonian(L, bL, cL, fp=32).info()
    from reapers_amd import proposer
    sched = ra.Schedule.from_mlp(proposer.load_weights())

    def run(nsteps, use_sched=True):
        return ra.syk_block_npoint(N, "otoc", sp=k, seed=seed, state_seed=seed + 1, beta=beta,
                                   tmax=tmax, nsteps=nsteps, krylov_dim=20, tol=1e-7, fp=32,
                                   schedule=sched if use_sched else None)

    # warm-up and the fixed part (E0, shift, pre-evolution, the t = 0 point)
    _, _, _, st0 = run(0)
    hip = ra.hip()
    ra.check(hip.rp_prof_reset())
    ra.check(hip.rp_prof_enable(1))
    t, v, e0, st = run(args.steps)
    n_ap, ms_ap = _prof_query(ra, ra.RP_KERNEL_APPLY)
    ra.check(hip.rp_prof_enable(0))
    per_point = (st.wall_ms - st0.wall_ms) / 1e3 / max(args.steps, 1)
    # the FP64 counterpart on the same couplings and initial state
    _, v64, _, _ = ra.syk_block_npoint(N, "otoc", sp=k, seed=seed, state_seed=seed + 1, beta=beta,
                                       tmax=tmax, nsteps=args.steps, krylov_dim=20, tol=1e-12,
                                       fp=64, promote=True)
    err64 = float(np.abs(v - v64).max())
    log("block OTOC FP32 vs promoted FP64: %.2e" % err64)
    fixed = None
    if not args.no_fixed:
        _, _, _, sf0 = run(0, False)
        _, vf, _, sf = run(args.steps, False)
        fixed = {"s_per_point": round((sf.wall_ms - sf0.wall_ms) / 1e3 / max(args.steps, 1), 4),
                 "matvecs": int(sf.matvecs), "max_abs_diff_F": float(np.abs(vf - v).max())}
    apply_ms = ms_ap / max(n_ap, 1)
    print(json.dumps({
        "mode": "block",
        "metric": "parity-block OTOC wall time per time point (sparse SYK N=48, beta=1)",
        "value": round(per_point, 4), "unit": "s",
        "fixed_part_s": round(st0.wall_ms / 1e3, 4),
        "t": [float(x) for x in t], "F": [[float("%.8g" % x.real), float("%.8g" % x.imag)] for x in v],
        "E0": e0, "matvecs": int(st.matvecs), "restarts": int(st.restarts),
        "rejected_proposals": int(st.rejected), "fixed_dim_20": fixed,
        "err_vs_fp64": err64,
        "config": {"workload": "sparse SYK k=8 N=48 in parity blocks (2 x 23 qubits), OTOC of "
                               "ops[N-2].LR, E0 shift, beta/8 pre-evolution, FP32 states, FP64 "
                               "reductions, proposer-chosen Krylov dims (fallback 20) tol 1e-7",
                   "terms_per_block": int(info.nterms),
                   "beta": beta, "tmax": tmax, "nsteps": args.steps, "seed": seed},
        "roofline": dict(apply_roofline(info, apply_ms, L, "apply_c64_syk46_traffic.json"),
                         launches=int(n_ap)),
    }), flush=True)


def ed_mode(ra, args):
    print(json.dumps(ed_result(ra, args, cpu=not args.no_cpu_baseline)), flush=True)


def ed_result(ra, args, cpu=True):
    """Dense SYK N=24 (12 qubits, 10626 strings) in FP64: restarted Krylov
    (dim 30, tol 1e-12) against exact diagonalization on the GPU at
    t in {0.5, 1, 2, 5}.  ED = dense build + rocSOLVER heevd once, then per t
    exp(-iHt) = V diag(e) V^H (one zgemm, 8 n^3 flops) and a gemv.
    value = Krylov wall time summed over the four t; the zgemm's roofline is
    taken from the wall time of the exponential of a new t (the zgemm's own
    kernel time is in the rocprof summary)."""
    N, L = 24, 12
    n = 1 << L
    times = [0.5, 1.0, 2.0, 5.0]
    bits, coeff = ra.syk_terms(N, 0.0, seed=args.seed, fp=64)
    H = ra.Hamiltonian(L, bits, coeff, fp=64)
    psi = ra.DeviceState(L, fp=64)
    psi.random(args.seed + 1)
    psi_host = psi.store()
    ed = ra.DeviceState(L, fp=64)
    kr = ra.DeviceState(L, fp=64)
    hip = ra.hip()
    # first ED call: dense build + eigensystem + first exponential
    ed.load(psi_host)
    ra.check(hip.rp_synchronize())
    t0 = time.perf_counter()
    ed.evolve_ed(H, 0.25)
    ra.check(hip.rp_synchronize())
    t_first = time.perf_counter() - t0
    rows = []
    kry_total = 0.0
    for t in times:
        ed.load(psi_host)
        ra.check(hip.rp_synchronize())
        t0 = time.perf_counter()
        ed.evolve_ed(H, t)
        ra.check(hip.rp_synchronize())
        t_ed = time.perf_counter() - t0
        kr.load(psi_host)
        kr.evolve(H, t, 0.0, krydim=30, tol=1e-12)          # warm-up
        kr.load(psi_host)
        ra.check(hip.rp_synchronize())
        t0 = time.perf_counter()
        st = kr.evolve(H, t, 0.0, krydim=30, tol=1e-12)
        ra.check(hip.rp_synchronize())
        t_kr = time.perf_counter() - t0
        kry_total += t_kr
        a, b = ed.store(), kr.store()
        rows.append({"t": t, "err_krylov_vs_ed": float(np.linalg.norm(a - b)),
                     "krylov_s": round(t_kr, 5), "krylov_matvecs": int(st.matvecs),
                     "ed_matexp_s": round(t_ed, 5)})
        log("t=%g: |krylov - ed| = %.2e, krylov %.4fs (%d matvecs), ED %.4fs" % (
            t, rows[-1]["err_krylov_vs_ed"], t_kr, st.matvecs, t_ed))
    # one new exponential (scaling kernel + zgemm) and the gemv, wall-clocked
    flops = 8.0 * n ** 3
    ed.load(psi_host)
    ra.check(hip.rp_synchronize())
    t0 = time.perf_counter()
    ed.evolve_ed(H, 7.5)
    ra.check(hip.rp_synchronize())
    t_new = time.perf_counter() - t0
    achieved = flops / t_new / 1e12
    peak = 78.6
    cpu_line = None
    if cpu:
        from oracle import krylov_evolve, num_threads
        t0 = time.perf_counter()
        out, _ = krylov_evolve(L, bits, coeff, psi_host, times[0], 0.0, krydim=30, tol=1e-12, fp=64)
        cpu_s = time.perf_counter() - t0
        ed.load(psi_host)
        ed.evolve_ed(H, times[0])
        cpu_line = {"value": round(cpu_s, 3), "unit": "s per exp(-iHt)psi at t=0.5", "cores": num_threads(),
               "kind": "port", "sample": "the whole t=0.5 evolution (oracle restatement of the "
                                         "reference's CPU Krylov, FP64, dim 30, tol 1e-12)",
               "err_vs_gpu_ed": float(np.linalg.norm(out - ed.store()))}
    for st_ in (H, psi, ed, kr):
        st_.close()
    return {
        "mode": "ed",
        "metric": "restarted Krylov vs GPU exact diagonalization, dense SYK N=24 (12 qubits), FP64",
        "value": round(kry_total, 5), "unit": "s (Krylov, four t)",
        "ed_first_call_s": round(t_first, 4), "rows": rows,
        "max_err_krylov_vs_ed": max(r["err_krylov_vs_ed"] for r in rows),
        "config": {"workload": "dense SYK q=4 N=24 (C(24,4)=10626 strings, dim 4096), seeded "
                               "Gaussian state, FP64, Krylov dim 30 tol 1e-12, t in {0.5,1,2,5}",
                   "terms": int(len(bits)), "seed": args.seed},
        "roofline": {"bound": "mfma", "achieved": round(achieved, 2), "peak": peak,
                     "unit": "TFLOP/s", "frac": round(achieved / peak, 4),
                     "kernel": "rocBLAS zgemm n=4096 in exp(-iHt) (wall time of the whole "
                               "uncached matexp + gemv)", "flops": flops,
                     "matexp_s": round(t_new, 5)},
        "cpu_baseline": cpu_line,
    }


def config_lines(ra, args):
    """The other benchmark configurations, each in a short form on its own
    workload (an error is recorded in place of its line): 1, dense SYK N=24
    in FP64, Krylov against exact diagonalization; 3, 64 sparse SYK
    realizations x 4 states in one batch; 5, the trained proposer on
    unseen XXZ L=26 and SYK N=48 (4, the N=60 OTOC point, runs with the
    30-qubit apply)."""
    out = {}
    for key, fn in (("3", lambda: batch_result(ra, single=False)),
                    ("5", lambda: proposer_result(ra)),
                    ("1", lambda: ed_result(ra, args, cpu=False))):
        t0 = time.perf_counter()
        try:
            out[key] = fn()
        except Exception as e:      # recorded, not fatal to the headline line
            out[key] = {"error": "%s: %s" % (type(e).__name__, e)}
        log("configuration %s: %.1fs" % (key, time.perf_counter() - t0))
    return out


def batched_n48(ra, args, bits, coeff, L, fp64_plain):
    """Four states sharing the N=48 Hamiltonian in one batch (the batch's
    autotuner times the batched apply, which stages each input tile once for
    all four states, against the plane apply, which runs the single-state
    kernel on each state), group accumulation, every restart's Krylov
    dimension from the trained proposer (fallback 20, at most 24), graph-
    replayed restarts; seconds per right-hand side against the plain FP64
    single-state Krylov, and each state's error against an FP64 evolution."""
    from reapers_amd import proposer
    nrhs, kmax = 4, 24
    states = []
    for q in range(nrhs):
        s = ra.DeviceState(L, fp=32)
        s.random(args.seed + 1 + q)
        states.append(s.store())
        s.close()
    block = np.stack(states, 1)
    b = ra.Batch([L], [(bits, coeff)], nrhs=nrhs, kmax=kmax, fp=32, autotune=True,
                 acc_group=True)
    sched = ra.Schedule.from_mlp(proposer.load_weights(), max_dim=kmax)
    b.load([block])
    b.evolve(args.t, m=args.krydim, tol=args.tol, schedule=sched)     # warm-up, graph capture
    hip = ra.hip()
    reps = 3
    t_total = 0.0
    for _ in range(reps):
        b.load([block])
        ra.check(hip.rp_synchronize())
        t0 = time.perf_counter()
        st, rs = b.evolve(args.t, m=args.krydim, tol=args.tol, schedule=sched)
        ra.check(hip.rp_synchronize())
        t_total += time.perf_counter() - t0
    per_batch = t_total / reps
    got = b.store()[0]
    info = b.info
    b.close()
    sched.close()
    errs = []
    H64 = ra.Hamiltonian(L, bits, coeff, fp=64)
    s64 = ra.DeviceState(L, fp=64)
    for q in range(nrhs):
        s64.load(states[q].astype(np.complex128))
        s64.evolve(H64, args.t, 0.0, krydim=args.krydim, tol=1e-13)
        ref = s64.store()
        errs.append(float(np.linalg.norm(got[:, q] - ref) / np.linalg.norm(ref)))
    s64.close()
    H64.close()
    per_rhs = per_batch / nrhs
    log("batched N=48: %d states in %.4f s (%.4f s per state), max err %.2e" % (
        nrhs, per_batch, per_rhs, max(errs)))
    return {
        "states": nrhs, "s_per_batch": round(per_batch, 5), "s_per_rhs": round(per_rhs, 5),
        "speedup_vs_fp64_plain": None if fp64_plain is None else round(fp64_plain / per_rhs, 3),
        "max_err_vs_fp64": max(errs), "restarts_max": int(rs.max()),
        "matvecs_per_rhs": int(st.matvecs) // nrhs if st.matvecs > nrhs else int(st.matvecs),
        "tiling": {"tile_bits": int(info.tile_bits), "threads": int(info.threads),
                   "planes": int(info.planes)},
        "workload": "4 seeded states x the same sparse SYK N=48 H, exp(-iHt) to t=%g, tol %g, "
                    "proposer-chosen Krylov dims (fallback %d, max %d), FP32 states with group "
                    "accumulation, FP64 reductions" % (args.t, args.tol, args.krydim, kmax),
    }


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--N", type=int, default=48)
    ap.add_argument("--k", type=float, default=8.0)
    ap.add_argument("--t", type=float, default=10.0)
    ap.add_argument("--krydim", type=int, default=20)
    ap.add_argument("--tol", type=float, default=1e-7)
    ap.add_argument("--seed", type=int, default=2000)
    ap.add_argument("--cpu-seconds", type=float, default=12.0)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-fp64", action="store_true")
    ap.add_argument("--no-batched", action="store_true",
                    help="skip the four-state batch sharing the N=48 Hamiltonian")
    ap.add_argument("--no-n60", action="store_true",
                    help="skip the 30-qubit apply measurement (8.6 GB states)")
    ap.add_argument("--schedule", choices=["mlp", "fixed"], default="mlp",
                    help="Krylov dimension per restart: the trained proposer (default) or "
                         "the fixed --krydim")
    ap.add_argument("--mode", choices=["evolve", "apply", "batch", "otoc", "proposer", "block",
                                       "ed"],
                    default="evolve",
                    help="apply: time only the Pauli-sum apply (both precisions), "
                         "for kernel profiling; batch: 64 sparse SYK realizations of "
                         "N in {32,36,40,44} x 4 states in one batch; otoc: N=60 OTOC points; "
                         "block: the parity-block OTOC driver at N=48; ed: Krylov vs GPU "
                         "exact diagonalization at N=24")
    ap.add_argument("--no-fixed", action="store_true",
                    help="otoc/block modes: skip the fixed-dimension comparison run")
    ap.add_argument("--apply-fp", choices=["32", "64", "both"], default="both",
                    help="apply mode: which state precisions to time")
    ap.add_argument("--no-autotune", action="store_true",
                    help="upload with the default tiling (no tiling trials)")
    ap.add_argument("--no-configs", action="store_true",
                    help="skip the short runs of the other configurations (1, 3, 4, 5)")
    ap.add_argument("--otoc-points", type=int, default=2,
                    help="otoc mode: how many of the 20 log-spaced times to evaluate")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU only: this build runs the whole state on one "
              "MI355X; --gpus %d is not supported" % args.gpus, file=sys.stderr)
        sys.exit(2)

    import reapers_amd as ra
    ra.init(0)
    # every Hamiltonian upload times the apply tilings and keeps the fastest;
    # complex<float> applies sum each tile group in FP32 and the groups in FP64
    ra.set_upload_flags((0 if args.no_autotune else ra.RP_TERMS_AUTOTUNE) | ra.RP_TERMS_ACC_GROUP)
    if args.mode == "batch":
        batch_mode(ra, args)
        return
    if args.mode == "otoc":
        otoc_mode(ra, args)
        return
    if args.mode == "proposer":
        proposer_mode(ra, args)
        return
    if args.mode == "block":
        block_mode(ra, args)
        return
    if args.mode == "ed":
        ed_mode(ra, args)
        return
    N, L = args.N, args.N // 2
    dim = 1 << L
    t_gen = time.perf_counter()
    bits, coeff = ra.syk_terms(N, args.k, seed=args.seed, fp=32)
    log("generated %d terms in %.2fs" % (len(bits), time.perf_counter() - t_gen))
    H32 = ra.Hamiltonian(L, bits, coeff, fp=32)
    info = H32.info()
    log("apply layout: tile_bits=%d flips=%d groups=%d bytes/apply=%.3e" % (
        info.tile_bits, info.nflips, info.ngroups, info.bytes_per_apply))

    psi0 = ra.DeviceState(L, fp=32)
    psi0.random(args.seed + 1)
    if args.mode == "apply":
        apply_only(ra, args, bits, coeff, L, psi0)
        return
    work = ra.DeviceState(L, fp=32)

    # FP64 reference of the same promoted Hamiltonian and state (untimed)
    err = None
    fp64_plain = None
    if not args.no_fp64:
        H64 = ra.Hamiltonian(L, bits, coeff, fp=64)
        ref = ra.DeviceState(L, fp=64)
        ref.copy_from(psi0)
        st_ref = ref.evolve(H64, args.t, 0.0, krydim=args.krydim, tol=1e-13)
        log("fp64 reference: %d matvecs %.3fs" % (st_ref.matvecs, st_ref.wall_ms / 1e3))
        # plain FP64 single-state Krylov at the target accuracy (the 3x denominator)
        w64 = ra.DeviceState(L, fp=64)
        w64.copy_from(psi0)
        st64 = w64.evolve(H64, args.t, 0.0, krydim=args.krydim, tol=1e-7)
        w64.copy_from(psi0)
        ra.check(ra.hip().rp_synchronize())
        t0 = time.perf_counter()
        st64 = w64.evolve(H64, args.t, 0.0, krydim=args.krydim, tol=1e-7)
        fp64_plain = time.perf_counter() - t0
        log("plain fp64: %d matvecs %.4fs" % (st64.matvecs, fp64_plain))
        w64.close()

    sched = None
    if args.schedule == "mlp":
        from reapers_amd import proposer
        sched = ra.Schedule.from_mlp(proposer.load_weights())

    def evolve32(w, use_sched=True):
        if sched is not None and use_sched:
            return w.evolve_with(H32, args.t, sched, krydim=args.krydim, tol=args.tol)
        return w.evolve(H32, args.t, 0.0, krydim=args.krydim, tol=args.tol)

    # FP32 with the fixed dimension (untimed warmup, then one timed run)
    fixed32 = None
    if sched is not None:
        work.copy_from(psi0)
        evolve32(work, False)
        work.copy_from(psi0)
        ra.check(ra.hip().rp_synchronize())
        t0 = time.perf_counter()
        stf = evolve32(work, False)
        fixed32 = {"s": round(time.perf_counter() - t0, 5), "matvecs": int(stf.matvecs),
                   "restarts": int(stf.restarts)}
        if not args.no_fp64:
            got = work.store().astype(np.complex128)
            want = ref.store()
            fixed32["err_vs_fp64"] = float(np.linalg.norm(got - want) / np.linalg.norm(want))
        log("fp32 fixed dim %d: %s" % (args.krydim, fixed32))

    for _ in range(args.warmup):
        work.copy_from(psi0)
        evolve32(work)

    hip = ra.hip()
    import ctypes
    # the timed region brackets only the apply launches with HIP events (the
    # roofline's kernel duration); bracketing every launch would add ~4% of
    # event overhead to the step time
    ra.check(hip.rp_prof_reset())
    ra.check(hip.rp_prof_enable(0x100 | (1 << ra.RP_KERNEL_APPLY)))
    ra.check(hip.rp_synchronize())
    t0 = time.perf_counter()
    stats = []
    for _ in range(args.steps):
        work.copy_from(psi0)
        stats.append(evolve32(work))
    ra.check(hip.rp_synchronize())
    elapsed = time.perf_counter() - t0
    n_apply, ms_apply = ctypes.c_uint64(), ctypes.c_double()
    ra.check(hip.rp_prof_query(ra.RP_KERNEL_APPLY, ctypes.byref(n_apply), ctypes.byref(ms_apply)))
    # per-class kernel times from one more (untimed) step with every launch bracketed
    ra.check(hip.rp_prof_reset())
    ra.check(hip.rp_prof_enable(1))
    work.copy_from(psi0)
    evolve32(work)
    ra.check(hip.rp_synchronize())
    n_gs, ms_gs = ctypes.c_uint64(), ctypes.c_double()
    ra.check(hip.rp_prof_query(ra.RP_KERNEL_GS, ctypes.byref(n_gs), ctypes.byref(ms_gs)))
    n_ot, ms_ot = ctypes.c_uint64(), ctypes.c_double()
    ra.check(hip.rp_prof_query(ra.RP_KERNEL_OTHER, ctypes.byref(n_ot), ctypes.byref(ms_ot)))
    ra.check(hip.rp_prof_enable(0))
    per_step = elapsed / args.steps
    matvecs = stats[-1].matvecs
    dims_used = None
    if sched is not None:
        sched.tracing(True)
        work.copy_from(psi0)
        evolve32(work)
        _, meta, _ = sched.trace()
        dims_used = [int(v) for k, v, _, _ in meta if k == 1]
        sched.tracing(False)

    if not args.no_fp64:
        got = work.store().astype(np.complex128)
        want = ref.store()
        err = float(np.linalg.norm(got - want) / np.linalg.norm(want))
        log("fp32 error vs fp64: %.3e" % err)

    avg_apply_ms = ms_apply.value / max(n_apply.value, 1)
    term_apps = info.nterms * dim / (avg_apply_ms / 1e3)
    roofline = apply_roofline(info, avg_apply_ms, L, "apply_c64_syk48_traffic.json")
    roofline["workload"] = ("sparse SYK k=8 N=48, 24 qubits, %d terms, complex<float> (the 128 MiB "
                            "state stays in the 256 MB Infinity Cache)" % info.nterms)
    batched = None
    if not args.no_batched:
        batched = batched_n48(ra, args, bits, coeff, L, fp64_plain)
    configs = None
    if not args.no_n60:
        roofline["n60"], otoc = n60_apply(ra, otoc_point=not args.no_configs)
        if otoc is not None:
            configs = {"4": otoc}
    if not args.no_configs:
        configs = configs or {}
        configs.update(config_lines(ra, args))
    line = {
        "metric": METRIC,
        "value": round(per_step, 5),
        "unit": "s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(per_step * 1e3, 3),
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "fp32",
        "data": "synthetic",
        "config": {
            "workload": "sparse SYK q=4 N=48 k=8, exp(-iHt)psi to t=%g, %s, "
                        "FP32 states + FP64 reductions/Hessenberg exp" % (
                            args.t, "proposer-chosen Krylov dims (fallback %d)" % args.krydim
                            if sched is not None else "Krylov dim %d" % args.krydim),
            "schedule": args.schedule,
            "N": N, "qubits": L, "dim": dim, "k": args.k, "terms": int(info.nterms),
            "t": args.t, "krydim": args.krydim, "tol": args.tol, "seed_H": args.seed,
            "seed_psi": args.seed + 1, "parallelism": "single GPU",
        },
        "err_vs_fp64": err,
        "matvecs_per_step": int(matvecs),
        "restarts_per_step": int(stats[-1].restarts),
        "gs_passes_per_step": int(stats[-1].gs_passes),
        "krylov_dims": dims_used,
        "rejected_proposals": int(stats[-1].rejected),
        "fp32_fixed_dim": fixed32,
        "fp64_plain_s": None if fp64_plain is None else round(fp64_plain, 5),
        "speedup_vs_fp64_plain": None if fp64_plain is None else round(fp64_plain / per_step, 3),
        "term_apps_per_s": float("%.4g" % term_apps),
        "apply_ms_per_step": round(ms_apply.value / args.steps, 3),
        "gs_ms_per_step": round(ms_gs.value, 3),
        "other_ms_per_step": round(ms_ot.value, 3),
        "roofline": roofline,
        "batched": batched,
        "configs": configs,
    }
    if not args.no_cpu_baseline:
        psi_host = psi0.store()
        line["cpu_baseline"] = cpu_baseline(bits, coeff, L, psi_host, matvecs, args.cpu_seconds)
    else:
        line["cpu_baseline"] = None
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
