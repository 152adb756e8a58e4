"""Benchmark: RHF time-to-solution and ERI quartets/s on one MI355X, plain
FP64 against mixed precision + learned guess, with the CPU oracle timed
beside it.

Workload (default, the headline): linear C20H42 in 6-31G* with Cartesian d
(384 basis functions), ideal zig-zag geometry with seeded Gaussian jitter
sigma = 0.02 A (seed 20010).  One step = one complete plain-FP64 RHF solve
from the geometry: Molecule, basis upload, S/T/V, Schwarz bounds, screened
ERIs into HBM (threshold 1e-8), SAD guess (atomic densities from the table
the library's atomic SCF made), SCF with Pulay DIIS to |dE| < 1e-10, final
orbitals.

Prints ONE JSON line.  ``value`` = screened unique ERI shell quartets per
second of whole-solve wall time.  Beside it:

* ``mixed_learned``: the same molecule with FP32 ERIs below a Schwarz bound
  product of 1e-6 and the learned (MLP) guess: time, speed-up over plain
  FP64, |dE| against it.
* ``roofline``: the J/K digestion class with the most time per solve, timed
  live in every Fock build of the timed solves (from its first block's start
  to its last block's end, by the GPU's realtime clock), against 8 TB/s;
  ``traffic`` from the rocprofv3 FETCH_SIZE / WRITE_SIZE runs summarised in
  profiles/pmc_traffic.json when they were taken for that kernel and
  workload; ``roofline.jk_build``: every class's digestion bytes over the
  time of a whole J/K build (all classes and the ket-J reduction).
* ``eri_roofline``: the ERI pass against the FP64 vector peak, flops priced
  as the reference prices them, Boys evaluations counted separately.
* ``config2``: C10H22 RHF + MP2 (FP64 and split-BF16 transforms).
* ``batch``: 512 molecules of uneven size in one batched RHF.
* ``cpu_baseline``: the oracle (oracle/oracle.c, OpenMP) on the host cores
  for the same C20H42 solve, from timed samples of the screened quartet list
  (see cpu_baseline()).

    python bench.py [--steps K] [--warmup W] [--gpus 1] [--no-cpu] [--no-batch] [--workload c20h42|c10h22|...]
    python bench.py --copy-calibration MIB   # plain device copy, for PMC byte-counter calibration
    python bench.py --only-rhf --steps 2     # plain RHF solves and the roofline only (profiling runs)
    python bench.py --jk-classes             # every J/K class timed alone on the converged density
    python bench.py --mp2 --workload c10h22  # the MP2 transform (FP64, BF16x3) on the converged RHF
"""
import argparse
import json
import os
import statistics
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

FP64_PEAK_TFLOPS = 78.6       # MI355X dense FP64 vector and FP64 matrix
HBM_PEAK_GBS = 8000.0

_ROWS = {}


def workload(name):
    """The workload's Molecule (built from its input rows on every call, as a
    solve starts) and its config.  The synthetic coordinates themselves are
    made once per workload: they are the input, not part of the solve."""
    from pychem_amd import geometry, structures
    if name == "water":
        return structures.Molecule(geometry.water(), basis="STO-3G"), {"workload": "H2O/STO-3G RHF", "nbf": 7}
    n = {"c4h10": 4, "c6h14": 6, "c8h18": 8, "c10h22": 10, "c14h30": 14, "c20h42": 20}[name]
    seed = 1000 * n + 10
    if name not in _ROWS:
        _ROWS[name] = geometry.alkane(n, 0.02, seed)
    rows = [list(r) for r in _ROWS[name]]
    mol = structures.Molecule(rows, basis="6-31G*", cartesian_l=[2])
    return mol, {"workload": "C%dH%d/6-31G* (6d) RHF, conv 1e-10" % (n, 2 * n + 2),
                 "nbf": mol.NOrbitals, "jitter_A": 0.02, "seed": seed}


def flop_model():
    with open(os.path.join(ROOT, "pychem_amd", "csrc", "eri_flops.json")) as fh:
        return json.load(fh)


def gpu_solve(name, timing=True, guess_kind="SAD", fp32_threshold=0.0, keep=False):
    """One whole solve; returns (result, class stats, per-class J/K times)."""
    from pychem_amd import guess, hartree_fock, structures
    guess._ATOM_CACHE.clear()          # no per-process cache carried between solves
    structures._SHELL_LAYOUTS.clear()
    mol = workload(name)[0]
    r = hartree_fock.run(mol, conv=1e-10, maxiter=100, timing=timing, guess=guess_kind,
                         fp32_threshold=fp32_threshold)
    stats = mol.Engine.stats()
    jkt = mol.Engine.jk_class_times() if timing else None
    if keep:
        return r, stats, jkt, mol
    mol.Engine.close()
    return r, stats, jkt


def jk_class_bytes(s, nitems, fm):
    """Algorithmic HBM bytes of one J/K digestion launch of a class: stored
    ERI values (8 B FP64, 4 B FP32 per component), the packed ket records
    (4 B per quartet), the work items (16 B, +8 B with an FP32 list) and the
    ket J values written (one per quartet, bra tile and ket component)."""
    la, lb, lc, ld = (int(x) for x in s["cls"])
    ta, tb, nt = fm[s["cls"]]["jk_tile"]
    ncd = (lc + 1) * (lc + 2) // 2 * ((ld + 1) * (ld + 2) // 2)
    nq = s["nq64"] + s["nq32"]
    return (s["nq64"] * s["ncomp"] * 8 + s["nq32"] * s["ncomp"] * 4 + nq * 4 +
            nitems * (16 + (8 if s["nq32"] else 0)) + nq * nt * ncd * 8)


def jk_kernel_name(cls, fm):
    """The class's part of its group's launch (jk_group_kernel_*)."""
    la, lb, lc, ld = (int(x) for x in cls)
    ta, tb, _ = fm[cls]["jk_tile"]
    return "jk_tile_class<%d, %d, %d, %d, %d, %d>" % (la, lb, lc, ld, ta, tb)


def pmc_traffic(kernel, workload_name):
    """HBM bytes per launch of ``kernel`` from the committed rocprofv3
    FETCH_SIZE / WRITE_SIZE summary (already scaled by the copy-kernel
    calibration), or None when it was taken for another kernel or workload."""
    path = os.path.join(ROOT, "profiles", "pmc_traffic.json")
    if not os.path.exists(path):
        return None
    with open(path) as fh:
        d = json.load(fh)
    if d.get("workload") != workload_name:
        return None
    for k in d.get("kernels", []):
        if k["kernel"] == kernel:
            return k["fetch_bytes"] + k["write_bytes"]
    return None


def copy_calibration(mib):
    """One plain device-to-device copy of ``mib`` MiB, repeated 5 times: the
    known-size reference for the PMC byte counters."""
    import torch
    n = mib * (1 << 20) // 8
    src = torch.ones(n, dtype=torch.float64, device="cuda")
    dst = torch.empty_like(src)
    for _ in range(5):
        dst.copy_(src)
    torch.cuda.synchronize()
    print(json.dumps({"copy_bytes_read": n * 8, "copy_bytes_written": n * 8, "launches": 5}))


def eri_model(stats, fm):
    """Algorithmic flops of one ERI pass priced as the reference prices them
    (VRR 6 per element, +5 with the a-term, +4 with the cross term;
    contraction 3; HRR 2 per contracted element), and the Boys evaluations
    (L + 1 values per primitive quartet), counted separately."""
    flops, boys = 0.0, 0.0
    for s in stats:
        f = fm[s["cls"]]
        nprim = s["nprim64"] + s["nprim32"]
        flops += (f["vrr"] + f["contract"]) * nprim + f["hrr"] * (s["nq64"] + s["nq32"])
        boys += f["boys"] * nprim
    return flops, boys


def mp2_measure(mol, r):
    """The MP2 transform (device events) in FP64 and with split-BF16
    products (FP32 accumulation) on the converged RHF; energies in FP64.
    Algorithmic flops of the O(N^5) quarter transforms and algorithmic bytes
    (the stored unique AO ERIs read once, the (ia|jb) block written)."""
    import torch
    from pychem_amd import mp2
    from pychem_amd.engine import mp2_energy
    eng = mol.Engine
    no = mol.NAlphaElectrons
    C, e = r["Ca"], r["ea"]
    n = C.shape[0]
    v = n - no
    flops = 2.0 * no * n ** 4 + 2.0 * no * v * n ** 3 + 2.0 * no * no * v * n ** 2 + 2.0 * no * no * v * v * n
    stored = sum(s["nq64"] * s["ncomp"] * 8 + s["nq32"] * s["ncomp"] * 4 for s in eng.stats())
    nbytes = stored + 8.0 * no * no * v * v
    res = {}
    for prec in ("fp64", "bf16x3"):
        mp2.run(mol, r, precision=prec)          # warm-up (allocations, code objects)
        t0 = torch.cuda.Event(enable_timing=True)
        t1 = torch.cuda.Event(enable_timing=True)
        t0.record()
        ov = eng.mp2_ovov(C[:, :no], C[:, no:], C[:, :no], C[:, no:], precision=prec)
        t1.record()
        ecorr = mp2_energy(ov, e[:no], e[no:], e[:no], e[no:], 0)
        torch.cuda.synchronize()
        ms = t0.elapsed_time(t1)
        del ov
        res[prec] = {"mp2_correlation": ecorr, "transform_ms": ms, "tflops": flops / (ms * 1e-3) / 1e12,
                     "gbs": nbytes / (ms * 1e-3) / 1e9}
    out = dict(res["fp64"], flops=flops, alg_bytes=nbytes, frac_fp64_peak=res["fp64"]["tflops"] / FP64_PEAK_TFLOPS,
               nocc=no, nvir=v)
    out["bf16x3"] = dict(res["bf16x3"], energy_error_vs_fp64=res["bf16x3"]["mp2_correlation"] -
                         res["fp64"]["mp2_correlation"],
                         speedup_vs_fp64=res["fp64"]["transform_ms"] / res["bf16x3"]["transform_ms"])
    return out


def config2_measure():
    """C10H22: plain FP64 RHF time and the MP2 transform rates."""
    import torch
    for _ in range(2):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        r, stats, _, mol = gpu_solve("c10h22", timing=False, keep=True)
        torch.cuda.synchronize()
        t_rhf = time.perf_counter() - t0
        if _ == 0:
            mol.Engine.close()
    nq = sum(s["nq64"] + s["nq32"] for s in stats)
    out = {"workload": workload("c10h22")[1]["workload"], "time_to_solution_s": t_rhf, "energy": r["energy"],
           "quartets_per_s": nq / t_rhf, "scf_iterations": r["iterations"], "mp2": mp2_measure(mol, r)}
    mol.Engine.close()
    return out


def batch_measure(count, steps):
    """512 molecules of uneven size (H2O, NH3, CH4, C2H6, CH3OH, C3H8 in STO-3G
    and 6-31G*, jitter 0.05 A, default_rng(4)) in one batched RHF; the J/K
    launch shapes come from the autotuner (tuned on an untimed pass)."""
    from pychem_amd.batch import config4_molecules, rhf_batch
    mols = config4_molecules(count, seed=4)
    warm = rhf_batch(mols, conv=1e-8, maxiter=80, tune="search")
    table = warm["tuned"]
    from pychem_amd import guess, structures
    runs = []
    for _ in range(max(1, steps)):
        ms = config4_molecules(count, seed=4)
        guess._ATOM_CACHE.clear()      # nothing carried over from the previous batch
        structures._SHELL_LAYOUTS.clear()
        runs.append(rhf_batch(ms, conv=1e-8, maxiter=80, tune=table))
    r = runs[-1]
    tot = float(np.median([x["total_s"] for x in runs]))
    lat = r["latency_s"]
    nbf = [m.NOrbitals for m in mols]
    return {"molecules": count, "nbf_min": int(min(nbf)), "nbf_max": int(max(nbf)),
            "molecules_per_s": count / tot, "wall_s": tot, "setup_s": r["setup_s"],
            "latency_p50_s": float(np.percentile(lat, 50)), "latency_p99_s": float(np.percentile(lat, 99)),
            "iterations_max": int(r["iterations"].max()), "all_converged": bool(r["converged"].all())}


def _cpu_model():
    try:
        with open("/proc/cpuinfo") as fh:
            for line in fh:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def _median_time(fn, reps):
    fn()                                   # warm-up
    ts = []
    for _ in range(reps):
        t0 = time.perf_counter()
        fn()
        ts.append(time.perf_counter() - t0)
    return statistics.median(ts)


def cpu_baseline(name, cycles, threads_all, reps=5):
    """The oracle's RHF of the same molecule on the host cores, from timed
    samples.  The dense (N^4) tensor of the reference does not fit at
    N = 384 (174 GB), so the oracle keeps the screened unique quartets as a
    list of final-basis blocks (or_eri_list) and digests them into J/K over
    their distinct 8-fold permutations (or_jk_list, equal to the dense
    einsums, tests/test_oracle.py).  Timed, per thread count (1 and all
    cores), median of ``reps`` runs after a warm-up: S/T/V, Schwarz bounds and
    the screening of every quartet in full; ERI generation and one J/K
    digestion on two systematic samples of the screened list (every 2048th
    and every 512th quartet), the per-quartet cost from their difference
    (which cancels the fixed per-call cost) times the full count, plus the
    fixed cost; per SCF cycle the J/K estimate and one eigh of X^T F X.
    Cycles: the GPU solve's count (the same SAD guess, Pulay DIIS and
    convergence test)."""
    from oracle import cint, scf as oscf
    mol = workload(name)[0]
    N = mol.NOrbitals
    legs = {}
    for th in (1, threads_all):
        cint.set_threads(th)
        t1e = _median_time(lambda: cint.one_electron(mol), reps)
        bounds = cint.schwarz(mol)
        tsch = _median_time(lambda: cint.schwarz(mol), reps)
        tot = [0]
        tscr = _median_time(lambda: tot.__setitem__(0, cint.screened_quartets(mol, bounds, 1e-8, stride=0)[0]),
                            max(1, reps // 2))
        total = tot[0]
        samples = {}
        D = np.eye(N) * 0.1
        for stride in (2048, 512):
            _, q = cint.screened_quartets(mol, bounds, 1e-8, stride=stride, offset=stride // 2)
            vals = cint.eri_list(mol, q)
            te = _median_time(lambda: cint.eri_list(mol, q), reps)
            tj = _median_time(lambda: cint.jk_list(mol, q, vals, D, D), reps)
            samples[stride] = (len(q), te, tj)
        (n1, e1, j1), (n2, e2, j2) = samples[2048], samples[512]
        pe, pj = max(0.0, (e2 - e1) / (n2 - n1)), max(0.0, (j2 - j1) / (n2 - n1))
        fe, fj = max(0.0, e1 - pe * n1), max(0.0, j1 - pj * n1)
        F = np.random.default_rng(0).normal(size=(N, N))
        F = F + F.T
        teig = _median_time(lambda: np.linalg.eigh(F), reps)
        t_eri = fe + pe * total
        t_jk = fj + pj * total
        t_solve = t1e + tsch + tscr + t_eri + cycles * (t_jk + teig)
        legs["%d_thread%s" % (th, "" if th == 1 else "s")] = {
            "threads": th, "one_electron_s": t1e, "schwarz_s": tsch, "screening_s": tscr,
            "eri_generation_s": t_eri, "eri_quartets_per_s": total / t_eri, "fock_build_s": t_jk,
            "fock_builds_per_s": 1.0 / t_jk, "eigh_s": teig, "scf_cycles": cycles,
            "time_to_solution_s": t_solve, "quartets_per_s": total / t_solve,
            "samples": {"every_2048th": {"quartets": n1, "eri_s": e1, "jk_s": j1},
                        "every_512th": {"quartets": n2, "eri_s": e2, "jk_s": j2}}}
    cint.set_threads(threads_all)
    return total, legs


FP32_MFMA_PEAK_TFLOPS = 157.3  # MI355X dense FP32 matrix


def mlp_measure(name, reps=10, batch=4096):
    """The learned guess's networks on the matrix cores (pq_mlp_forward /
    _backward, v_mfma_f32_16x16x4f32): the inference over every atom-pair group of
    the workload (what a solve with the learned guess runs) and one training
    step (forward and backward) of the largest network on a batch, each timed
    with HIP events on the working stream.  Flops: 2 B sum(in x out) per
    forward, three times that for forward plus backward."""
    import torch
    from pychem_amd import mlp_guess
    nets = mlp_guess.default_nets()
    if not nets:
        return None
    mol = workload(name)[0]
    groups = mlp_guess.pair_data(mol)
    inputs = []
    for key, (_, _, F, _) in groups.items():
        net = nets.get(key)
        if net is not None:
            inputs.append((net, torch.tensor(((F - net.xmean) / net.xstd).astype(np.float32), device="cuda")))
    if not inputs:
        return None

    def flops(net, B):
        return 2.0 * B * sum(net.dims[i] * net.dims[i + 1] for i in range(4))

    def timed(fn):
        fn()
        torch.cuda.synchronize()
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(reps):
            fn()
        b.record()
        torch.cuda.synchronize()
        return a.elapsed_time(b) / reps

    inf_ms = timed(lambda: [net.forward(X) for net, X in inputs])
    inf_flop = sum(flops(net, X.shape[0]) for net, X in inputs)
    net = max(inputs, key=lambda t: t[1].shape[0])[0]
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    Xb = torch.randn((batch, net.dims[0]), generator=g, device="cuda")
    Tb = torch.randn((batch, net.dims[-1]), generator=g, device="cuda")

    def train_step():
        Y, acts = net.forward(Xb, keep=True)
        _, dY = net.loss_grad(Y, Tb)
        net.backward(acts, dY)

    tr_ms = timed(train_step)
    tr_flop = 3.0 * flops(net, batch)
    return {"bound": "mfma", "unit": "TFLOP/s", "peak": FP32_MFMA_PEAK_TFLOPS,
            "inference": {"pairs": int(sum(X.shape[0] for _, X in inputs)), "networks": len(inputs),
                          "ms": round(inf_ms, 4), "flop": inf_flop,
                          "achieved": round(inf_flop / (inf_ms * 1e-3) / 1e12, 4),
                          "frac": round(inf_flop / (inf_ms * 1e-3) / 1e12 / FP32_MFMA_PEAK_TFLOPS, 6)},
            "training_step": {"batch": batch, "dims": list(net.dims), "ms": round(tr_ms, 4), "flop": tr_flop,
                              "achieved": round(tr_flop / (tr_ms * 1e-3) / 1e12, 4),
                              "frac": round(tr_flop / (tr_ms * 1e-3) / 1e12 / FP32_MFMA_PEAK_TFLOPS, 6)}}


def jk_classes_measure(name, reps=10):
    """Every J/K class digested alone (pq_jk_class: the tiled digestion
    kernel, then the ket-side J reduction, each timed with HIP events on the
    working stream over ``reps`` launches) on the converged density, and the
    whole J/K build on 1 to 4 streams (the caller's one of them)."""
    import ctypes
    import torch
    from pychem_amd import _lib
    from pychem_amd.engine import _ptr, _stream
    from pychem_amd._lib import check
    r, stats, _, mol = gpu_solve(name, timing=False, keep=True)
    eng = mol.Engine
    fm = flop_model()
    n = eng.ncart
    D = eng.to_cart(torch.as_tensor(r["Da"]).to(eng.device)).contiguous()
    J = torch.zeros((n, n), dtype=torch.float64, device=eng.device)
    K = torch.zeros_like(J)
    L = _lib.lib()

    def ev_time(fn):
        fn()
        torch.cuda.synchronize()
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(reps):
            fn()
        b.record()
        torch.cuda.synchronize()
        return a.elapsed_time(b) / reps

    rows = []
    for s in stats:
        c = s["index"]
        if s["nq64"] + s["nq32"] == 0:
            continue
        nit = ctypes.c_int()
        check(L.pq_jk_class(eng.h, c, 3, _ptr(D), _ptr(D), _ptr(J), _ptr(K), ctypes.byref(nit), _stream()), "pq_jk_class")
        part = lambda p: (lambda: check(L.pq_jk_class(eng.h, c, p, _ptr(D), _ptr(D), _ptr(J), _ptr(K), None,
                                                      _stream()), "pq_jk_class"))
        t1, t2 = ev_time(part(1)), ev_time(part(2))
        b = jk_class_bytes(s, nit.value, fm)
        rows.append({"cls": s["cls"], "kernel": jk_kernel_name(s["cls"], fm), "quartets": s["nq64"] + s["nq32"],
                     "ncomp": s["ncomp"], "items": nit.value, "digest_ms": round(t1, 4), "reduce_ms": round(t2, 4),
                     "bytes": b, "digest_gbs": round(b / (t1 * 1e-3) / 1e9, 1)})
    streams = {}
    for ns in (1, 2, 3, 4):
        check(L.pq_jk_set_streams(eng.h, ns), "pq_jk_set_streams")
        streams[ns] = round(ev_time(lambda: eng.jk(D, D)), 4)
    check(L.pq_jk_set_streams(eng.h, 4), "pq_jk_set_streams")
    eng.close()
    return {"workload": workload(name)[1]["workload"], "classes": rows,
            "digest_ms_sum": round(sum(x["digest_ms"] for x in rows), 4),
            "reduce_ms_sum": round(sum(x["reduce_ms"] for x in rows), 4), "jk_ms_by_streams": streams}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--workload", default="c20h42")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--cpu-threads", type=int, default=0)
    ap.add_argument("--no-batch", action="store_true")
    ap.add_argument("--batch-size", type=int, default=512)
    ap.add_argument("--copy-calibration", type=int, default=0, metavar="MIB")
    ap.add_argument("--mp2", action="store_true",
                    help="the workload's RHF, then its MP2 transform in FP64 and BF16x3 (one JSON line)")
    ap.add_argument("--jk-classes", action="store_true",
                    help="time every J/K class alone on the workload's converged density (one JSON line)")
    ap.add_argument("--only-rhf", action="store_true",
                    help="plain RHF solves and the roofline only (no mixed, config-2, batch or CPU legs): "
                         "the command the per-kernel profiles are taken on")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU only: this build has no multi-GPU path (run with --gpus 1)",
              file=sys.stderr)
        sys.exit(2)

    import torch
    from pychem_amd import _lib
    if not torch.cuda.is_available():
        raise _lib.HipError("no GPU visible")
    if args.copy_calibration:
        copy_calibration(args.copy_calibration)
        return
    if args.jk_classes:
        print(json.dumps(jk_classes_measure(args.workload)))
        return
    if args.mp2:
        r, _, _, mol = gpu_solve(args.workload, timing=False, keep=True)
        out = {"workload": workload(args.workload)[1]["workload"], "mp2": mp2_measure(mol, r)}
        mol.Engine.close()
        print(json.dumps(out))
        return
    _lib.lib()
    cfg = workload(args.workload)[1]
    fm = flop_model()

    for _ in range(args.warmup):
        gpu_solve(args.workload)
    torch.cuda.synchronize()
    results = []
    step_ms = []
    t0 = time.perf_counter()
    for _ in range(args.steps):
        ts = time.perf_counter()
        results.append(gpu_solve(args.workload))
        step_ms.append(1e3 * (time.perf_counter() - ts))
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    ms_per_step = 1e3 * wall / args.steps
    r0, stats, _ = results[-1]
    nq = sum(s["nq64"] + s["nq32"] for s in stats)
    nprim = sum(s["nprim64"] + s["nprim32"] for s in stats)
    value = nq * args.steps / wall

    # the dominant J/K digestion class: the most time per solve, every Fock
    # build of the timed solves timed
    sums = sum(x[2][0] for x in results)
    launches = sum(x[2][1] for x in results)
    nitems = results[-1][2][2]
    per_class = []
    for s, ms, n, it in zip(stats, sums, launches, nitems):
        if n == 0:
            continue
        b = jk_class_bytes(s, int(it), fm)
        avg = ms / n
        per_class.append({"cls": s["cls"], "kernel": jk_kernel_name(s["cls"], fm), "launches": int(n),
                          "avg_ms": round(avg, 5), "ms_per_solve": round(ms / args.steps, 4), "bytes": int(b),
                          "gbs": round(b / (avg * 1e-3) / 1e9, 1)})
    dom = max(per_class, key=lambda c: c["ms_per_solve"])
    achieved = dom["bytes"] / (dom["avg_ms"] * 1e-3) / 1e9
    roofline = {"bound": "hbm", "kernel": dom["kernel"], "achieved": round(achieved, 2), "peak": HBM_PEAK_GBS,
                "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 5),
                "traffic": pmc_traffic(dom["kernel"], cfg["workload"]),
                "alg_bytes_per_launch": dom["bytes"], "avg_launch_ms": dom["avg_ms"],
                "launches_timed": dom["launches"], "ms_per_solve": dom["ms_per_solve"],
                "jk_classes": sorted(per_class, key=lambda c: -c["ms_per_solve"])}
    jk_ms = [x for r, _, _ in results for x in r["timings"]["jk_ms"]]
    jk_avg = float(np.mean(jk_ms)) if jk_ms else 0.0
    if jk_avg > 0:
        # the whole Fock build: every class's digestion bytes over the time of
        # one J/K (all classes on their streams plus the ket-J reduction)
        jb = sum(c["bytes"] for c in per_class)
        roofline["jk_build"] = {"alg_bytes": int(jb), "ms": round(jk_avg, 4),
                                "achieved": round(jb / (jk_avg * 1e-3) / 1e9, 2),
                                "frac": round(jb / (jk_avg * 1e-3) / 1e9 / HBM_PEAK_GBS, 5)}

    eri_pass_ms = float(np.mean([r["timings"]["eri_pass_ms"] for r, _, _ in results]))
    eflops, boys = eri_model(stats, fm)
    eri_roofline = {"bound": "fp64-valu", "kernel": "ERI pass (21 class kernels on 4 streams)",
                    "achieved": round(eflops / (eri_pass_ms * 1e-3) / 1e12, 4), "peak": FP64_PEAK_TFLOPS,
                    "unit": "TFLOP/s", "frac": round(eflops / (eri_pass_ms * 1e-3) / 1e12 / FP64_PEAK_TFLOPS, 5),
                    "alg_flop_per_pass": eflops, "boys_evaluations_per_pass": boys, "pass_ms": round(eri_pass_ms, 4),
                    "primitive_quartets": nprim}
    out = {
        "metric": "RHF time-to-solution & ERI quartets/s: plain FP64 vs mixed+learned, 1 GPU",
        "value": value, "unit": "ERI shell quartets/s (whole RHF solve)",
        "n_gpus": 1, "steps": args.steps, "warmup": args.warmup, "ms_per_step": ms_per_step,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f64",
        "data": "synthetic geometry (seeded jitter), reference basis data",
        "config": dict(cfg, threshold=1e-8, precision="plain FP64", guess="SAD"),
        "time_to_solution_s": ms_per_step / 1e3, "energy": r0["energy"], "scf_iterations": r0["iterations"],
        "quartets_per_solve": nq, "primitive_quartets_per_solve": nprim,
        "eri_pass_ms": eri_pass_ms, "fock_builds_per_s": 1e3 / jk_avg if jk_avg > 0 else None, "jk_ms": jk_avg,
        "stage_s": {k: v for k, v in r0["timings"].items() if isinstance(v, float)},
        "final_orbitals": r0["timings"].get("final_orbitals"),
        "orthogonaliser": r0["timings"].get("orthogonaliser"),
        "purify_steps": r0["timings"].get("purify_steps"),
        "late_eigh": [r["timings"].get("late_eigh") for r, _, _ in results],
        "step_ms": [round(x, 3) for x in step_ms],
        "roofline": roofline,
        "eri_roofline": eri_roofline,
    }
    if not args.only_rhf:
        # the headline pair: mixed precision + learned guess on the same molecule
        gpu_solve(args.workload, timing=False, guess_kind="MLP", fp32_threshold=1e-6)
        torch.cuda.synchronize()
        tm = time.perf_counter()
        mixed = [gpu_solve(args.workload, timing=False, guess_kind="MLP", fp32_threshold=1e-6)
                 for _ in range(args.steps)]
        torch.cuda.synchronize()
        mixed_s = (time.perf_counter() - tm) / args.steps
        rm, sm, _ = mixed[-1]
        out["mixed_learned"] = {"time_to_solution_s": mixed_s, "speedup_vs_plain_fp64": (ms_per_step / 1e3) / mixed_s,
                                "energy_error_vs_fp64": rm["energy"] - r0["energy"], "scf_iterations": rm["iterations"],
                                "guess": rm["timings"].get("guess_kind"),
                                "fp32_quartets": sum(s["nq32"] for s in sm), "fp64_quartets": sum(s["nq64"] for s in sm)}
        out["config2"] = config2_measure()
        out["mlp_roofline"] = mlp_measure(args.workload)
        if not args.no_batch:
            out["batch"] = batch_measure(args.batch_size, args.steps)
        if not args.no_cpu:
            ncores = args.cpu_threads or len(os.sched_getaffinity(0))
            total, legs = cpu_baseline(args.workload, r0["iterations"], ncores)
            allc = legs["%d_threads" % ncores] if ncores > 1 else legs["1_thread"]
            out["cpu_baseline"] = {
                "value": allc["quartets_per_s"], "unit": out["unit"], "cores": ncores, "kind": "port",
                "cpu_model": _cpu_model(),
                "sample": "oracle RHF of the same %s molecule from timed samples: S/T/V, Schwarz and screening of "
                          "all %d screened quartets in full; ERI generation and one J/K digestion on every 2048th "
                          "and every 512th screened quartet (per-quartet cost from the difference, times the full "
                          "count, plus the fixed cost); %d SCF cycles (the GPU solve's, same SAD guess) of J/K and "
                          "one eigh; median of 5 after a warm-up; 1 thread and %d threads" %
                          (args.workload, total, r0["iterations"], ncores),
                "time_to_solution_s": allc["time_to_solution_s"], "legs": legs}
            out["gpu_vs_cpu"] = value / out["cpu_baseline"]["value"]
            out["gpu_vs_cpu_1_thread"] = value / legs["1_thread"]["quartets_per_s"]
    print(json.dumps(out))


if __name__ == "__main__":
    main()
