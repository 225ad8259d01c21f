"""Benchmark: atom-steps/s of E + F + magnetic gradients for 16000-atom bcc Fe on one MI355X.

Workload (the configuration the headline metric is quoted on): bcc Fe 20x20x20 conventional
cells (16000 atoms, a = 2.83 A, periodic), positions jittered N(0, 0.05 A), ferromagnetic
spins along z with a random cone angle U[0, 30 deg], magnitudes N(2.2, 0.1) muB, r_c 5.0 A;
potential header "10 3 2 6 / 7 1 6 1 / 3 1 3 1" (lmax 6, nradmax 10, 2043 B functions),
coefficients N(0, 1e-2), seed 2028.  A step is one full evaluation (libace acelib_ semantics:
pair list prebuilt, inputs resident in HBM): energies, pair forces, pair and self magnetic
gradients.  The mixed path is the headline value; the FP64 path runs on the same inputs and
the mixed path's error against it is reported.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu]
"""
from __future__ import annotations

import argparse
import json
import os
import subprocess
import sys
import tempfile
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)
import __graft_entry__  # noqa: E402

SEED = 2028
PEAK = {"mixed": 157.3, "fp64": 78.6}  # TFLOP/s, MI355X published vector FP32 / FP64


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def measured_traffic(kernel):
    """HBM bytes per launch of a kernel on this workload, from the rocprofv3 FETCH_SIZE /
    WRITE_SIZE passes summarised in profiles/fe16k_lmax6_traffic.txt (scaled by the plain-copy
    calibration recorded there).  None if the summary is absent."""
    path = os.path.join(ROOT, "profiles", "fe16k_lmax6_traffic.txt")
    if not os.path.exists(path):
        return None
    for line in open(path):
        if line.startswith(kernel + " "):
            return int(dict(kv.split("=") for kv in line.split()[1:])["bytes"])
    return None


def mixed_traffic(kernel):
    """measured_traffic of the mixed-precision launch of a kernel ("density", "adjoint", "forces")."""
    return measured_traffic({"density": "k_density_mm", "adjoint": "k_adjoint_nodes", "forces": "k_forces_mm"}[kernel] + "<float>")


def md_leg(pkg, td, steps=100, warmup=20):
    """Secondary measurement: device-resident spin-lattice MD, 128000 bcc Fe atoms (40^3
    cells), lmax-4 header "8 3 2 4 / 4 1 4 1 / 2 1 2 1" with c ~ N(0, 1e-3) (seed 2030),
    displacements N(0, 0.063 A) (1000 K, omega = 61.5 rad/ps, Debye 470 K), Maxwell velocities
    at 1000 K, uniform spins, dt = 0.1 fs, list cutoff 5.5 A rebuilt every 10 steps on the
    device, steps replayed from a captured HIP graph, mixed precision."""
    capi, potgen, systems, md = pkg.capi, pkg.potgen, pkg.systems, pkg.md
    h = dict(potgen.H500)
    pot = os.path.join(td, "Fe_md.pbe.in")
    with open(pot, "w") as f:
        f.write(potgen.render(h, capi.enumerate_basis(h), 2030, c_scale=1e-3))
    capi.init_file(pot)
    capi.set_precision(capi.MIXED)
    rng = np.random.default_rng(2030)
    pos, cell = systems.bcc(40)
    pos = systems.jitter(pos, rng, 0.063)
    sdir, smag = systems.spins_uniform(len(pos), rng)
    vel = md.maxwell_velocities(len(pos), 1000.0, rng)
    m = md.SpinLatticeMD(pos, cell, sdir, smag, vel=vel, dt=1e-4, rcut=5.0, skin=0.5, rebuild_every=10)
    st0 = m.state()
    m.run(warmup)
    m.state()
    t0 = time.perf_counter()
    m.run(steps)
    st = m.state()
    dt = time.perf_counter() - t0
    m.close()
    n = len(pos)
    return {"workload": "spin-lattice MD, bcc Fe 40x40x40 (%d atoms), lmax-4 header (489 B functions), "
                        "1000 K, dt 0.1 fs, neighbour rebuild every 10 steps on the device, HIP graph" % n,
            "atoms": n, "steps": steps, "ms_per_step": 1e3 * dt / steps, "atom_steps_per_s": n * steps / dt,
            "pairs": st["pairs"], "rebuilds": st["rebuilds"] - st0["rebuilds"], "graph_captures": st["captures"],
            "energy_drift_per_atom": (st["epot"] + st["ekin"] - st0["epot"] - st0["ekin"]) / n}


def fit_leg(pkg, td, steps=5):
    """Secondary measurement: one batched fit step = energies and forces of 256 periodic bcc Fe
    configurations (14-1023 atoms, log-uniform sizes, strain +-3%, 0-2 vacancies; seed 2029)
    and the gradient of a loss in all 489 coefficients of the lmax-4 header (FP64): the
    device neighbour build runs once, each step is magace_fit_set_coefficients +
    magace_fit_forward + magace_fit_backward."""
    import torch
    capi, potgen, systems, fit = pkg.capi, pkg.potgen, pkg.systems, pkg.fit
    h = dict(potgen.H500)
    pot = os.path.join(td, "Fe_fit.pbe.in")
    with open(pot, "w") as f:
        f.write(potgen.render(h, capi.enumerate_basis(h), 2029))
    capi.init_file(pot)
    structs = systems.config_batch()
    t0 = time.perf_counter()
    batch = fit.Batch(structs, 5.0)
    torch.cuda.synchronize()
    t_nb = time.perf_counter() - t0
    dev = batch.device
    c = capi.fit_get_coefficients()
    E = torch.zeros(batch.nstruc, dtype=torch.float64, device=dev)
    F = torch.zeros(batch.natom, 3, dtype=torch.float64, device=dev)
    gE = torch.ones(batch.nstruc, dtype=torch.float64, device=dev)
    gF = torch.ones(batch.natom, 3, dtype=torch.float64, device=dev)
    g = torch.zeros(len(c), dtype=torch.float64, device=dev)

    def step():
        # as an optimiser step runs it: new coefficients (merged weights recomputed and
        # uploaded), forward, backward
        capi.fit_set_coefficients(c)
        batch.forward(E, F)
        batch.backward(gE, gF, g)

    step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        step()
    torch.cuda.synchronize()
    dt = (time.perf_counter() - t0) / steps
    return {"workload": "batched fit step: 256 bcc Fe configurations (%d atoms, %d pairs), lmax-4 header, "
                        "coefficient upload + energies + forces + dL/dc (489 coefficients), FP64" % (batch.natom, batch.npairs),
            "configs": batch.nstruc, "atoms": batch.natom, "ms_per_step": 1e3 * dt,
            "atom_steps_per_s": batch.natom / dt, "configs_per_s": batch.nstruc / dt,
            "neighbour_build_s": t_nb}


def _sub(a, lo, hi):
    """acelib_ arrays of atoms [lo, hi) of a packed list (pair ranges re-based)."""
    off = a["offsets"]
    p0, p1 = int(off[lo]), int(off[hi])
    st = (a["nstart"][lo:hi] - p0).astype(np.int32)
    sp = (a["nstop"][lo:hi] - p0).astype(np.int32)
    return dict(nstart=st, nstop=sp, nlist=a["nlist"][p0:p1], occ=a["occ"][lo:hi], occlist=a["occlist"][p0:p1],
                dlist=a["dlist"][p0:p1], elist=a["elist"][3 * p0:3 * p1], dlist_momi=a["dlist_momi"][lo:hi],
                elist_momi=a["elist_momi"][3 * lo:3 * hi], dlist_mom=a["dlist_mom"][p0:p1],
                elist_mom=a["elist_mom"][3 * p0:3 * p1], nall=hi - lo)


def cpu_model():
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(pot, a, atoms_per_proc=100, nproc=None, nreps=5, single_atoms=400):
    """The reference libace (oracle/_ref: built from its Fortran sources, AMD flang -O2, serial)
    on the host cores, as LAMMPS runs it under MPI: nproc independent processes, each calling
    acelib_ on its own sub-range of atoms_per_proc atoms of the same workload (its pairs
    prebuilt), all at once.  Each process makes 1 warm-up and nreps timed calls; the rate is
    the sum over processes of atoms / median call time.  Beside it, one process on
    single_atoms atoms alone (1 core).  nproc defaults to the host's CPU share: at most 16
    cores.  Returns None if the reference binary is absent."""
    import concurrent.futures as cf
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle as O
    if not os.path.exists(O.REF_DRIVER):
        return None
    ncpu = os.cpu_count() or 1
    nproc = nproc or min(16, ncpu)
    drv = O.RefDriver(pot)
    t0 = time.perf_counter()
    one = drv.run(_sub(a, 0, single_atoms), nreps=1 + nreps, timeout=900)
    t1 = float(np.median(one["seconds"][1:]))
    single = dict(value=single_atoms / t1, cores=1, atoms=single_atoms, median_s=t1,
                  seconds=one["seconds"][1:].tolist())
    subs = [_sub(a, k * atoms_per_proc, (k + 1) * atoms_per_proc) for k in range(nproc)]
    with cf.ThreadPoolExecutor(max_workers=nproc) as ex:
        outs = list(ex.map(lambda sb: drv.run(sb, nreps=1 + nreps, timeout=900), subs))
    med = [float(np.median(o["seconds"][1:])) for o in outs]
    rate = sum(atoms_per_proc / m for m in med)
    log("cpu baseline: %.1f s wall" % (time.perf_counter() - t0))
    return {"value": rate, "unit": "atom-steps/s", "cores": nproc, "kind": "reference",
            "sample": "%d processes at once, each acelib_ on its own %d of the 16000 atoms (%d atoms, %d pairs "
                      "in all), reference libace built from its Fortran sources with AMD flang -O2 (serial), "
                      "1 warm-up + %d timed calls per process, rate = sum of atoms / median call time"
                      % (nproc, atoms_per_proc, nproc * atoms_per_proc,
                         int(a["offsets"][nproc * atoms_per_proc]), nreps),
            "warmup": 1, "nreps": nreps, "host_cpus": ncpu, "cpu_model": cpu_model(),
            "median_s_per_process": med, "single_core": single}


def oracle_errors(pot, a, outs, natom_sample=2000):
    """Per-output errors of the GPU outputs against the oracle (the C restatement of the
    reference, FP64, 16 threads) on the first natom_sample atoms of the workload: max |dE_i|,
    max |dF_p|, max |dT_p|, max |dT0_i| (eV, eV/A, eV/muB) per precision, and the FP64 path's
    norm-wise relative error per output array."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle as O
    S = natom_sample
    P = int(a["offsets"][S])
    ref = O.Oracle.load(pot).acelib(_sub(a, 0, S), nthreads=min(16, os.cpu_count() or 1))
    cut = dict(eout=S, flist=3 * P, tlist=3 * P, tlist0=3 * S)
    res = {"sample": "first %d atoms (%d pairs) of the 16000" % (S, P)}
    for prec, o in outs.items():
        res[prec] = {k: float(np.abs(o[k][:n] - ref[k]).max()) for k, n in cut.items()}
        res[prec + "_rel"] = {k: float(np.abs(o[k][:n] - ref[k]).max() / max(np.abs(ref[k]).max(), 1e-300))
                              for k, n in cut.items()}
    return res


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--ncell", type=int, default=20)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--cpu-sample", type=int, default=100,
                    help="atoms per reference process in the CPU baseline")
    ap.add_argument("--no-md", action="store_true",
                    help="skip the secondary legs (128000-atom spin-lattice MD, 256-configuration fit step)")
    ap.add_argument("--no-host-arrays", action="store_true",
                    help="skip the acelib_ timing on host arrays (its chunked launches would mix into "
                         "per-kernel profiles of the full-size launches)")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="first run one plain 512 MiB device copy (the reference kernel for HBM counters)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py: the evaluator runs on one GPU; a multi-GPU run (spatial decomposition "
              "with ghost exchange) is not implemented", file=sys.stderr)
        sys.exit(2)

    import torch
    assert torch.cuda.is_available(), "bench.py needs a GPU"
    dev = torch.device("cuda:0")
    pkg = __graft_entry__.load_package()
    capi, potgen, systems = pkg.capi, pkg.potgen, pkg.systems
    import importlib
    flops = importlib.import_module("magace_amd.flops")

    if args.calibrate_copy:
        src = torch.ones(64 << 20, dtype=torch.float64, device=dev)
        dst = torch.empty_like(src)
        dst.copy_(src)
        torch.cuda.synchronize()
        log("calibration copy: %d bytes read, %d bytes written" % (src.numel() * 8, dst.numel() * 8))
        del src, dst

    H = potgen.H2000
    td = tempfile.mkdtemp(prefix="magace_bench_")
    pot = os.path.join(td, "Fe.pbe.in")
    basis = capi.enumerate_basis(H)
    potgen.write(pot, H, basis, SEED)
    t0 = time.perf_counter()
    s = systems.make_system(args.ncell, SEED, spins="cone")
    a = systems.pack_acelib(s["pos"], s["cell"], s["sdir"], s["smag"], 5.0)
    N, P = int(a["natom"]), int(len(a["dlist"]))
    log("system: %d atoms, %d pairs (%.1f neighbours/atom), built in %.1f s" %
        (N, P, P / N, time.perf_counter() - t0))
    t0 = time.perf_counter()
    capi.init_file(pot)
    info = capi.model_info()
    log("init: %.2f s, %d monomials (from %d m-combinations), feature vector %d" %
        (time.perf_counter() - t0, info["terms"], info["raw"], info["nz"]))

    T = lambda x, dt=torch.float64: torch.as_tensor(np.ascontiguousarray(x), dtype=dt, device=dev)
    off = T(a["offsets"], torch.int32)
    ins = [T(a[k]) for k in ("dlist", "elist", "dlist_momi", "elist_momi", "dlist_mom", "elist_mom")]
    stream = torch.cuda.current_stream().cuda_stream

    def alloc():
        return [torch.zeros(N, dtype=torch.float64, device=dev), torch.zeros(3 * P, dtype=torch.float64, device=dev),
                torch.zeros(3 * P, dtype=torch.float64, device=dev), torch.zeros(3 * N, dtype=torch.float64, device=dev)]

    def step(outs):
        capi.compute_device(N, P, off.data_ptr(), *[x.data_ptr() for x in ins], *[x.data_ptr() for x in outs],
                            stream=stream)

    res = {}
    for prec, mode in (("fp64", capi.FP64), ("mixed", capi.MIXED), ("mixed_acc", capi.MIXED_ACC)):
        capi.set_precision(mode)
        outs = alloc()
        for _ in range(args.warmup):
            step(outs)
        capi.check_errors(stream)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.steps):
            step(outs)
        torch.cuda.synchronize()
        dt = time.perf_counter() - t0
        capi.check_errors(stream)
        # per-kernel times from a second pass with HIP events between the kernels; in this mode
        # an evaluation runs its atoms in one sequence, not as two overlapped halves
        capi.profile(True)
        for _ in range(args.steps):
            step(outs)
        torch.cuda.synchronize()
        kms, cnt = capi.profile_read()
        capi.profile(False)
        capi.check_errors(stream)
        res[prec] = dict(ms_per_step=1e3 * dt / args.steps, value=N * args.steps / dt,
                         kernel_ms=(kms / max(cnt, 1)).tolist(),
                         out={k: o.cpu().numpy() for k, o in zip(("eout", "flist", "tlist", "tlist0"), outs)})
        log("%s: %.3f ms/step, %.3e atom-steps/s, kernels [density, adjoint, forces] ms %s" %
            (prec, res[prec]["ms_per_step"], res[prec]["value"], np.round(kms / max(cnt, 1), 4).tolist()))

    # the boundary as LAMMPS uses it: acelib_ on host arrays (copies over PCIe included)
    # (output arrays kept between calls, as the caller keeps them between steps)
    host_ms = None
    if not args.no_host_arrays:
        capi.set_precision(capi.MIXED)
        host_out = capi.acelib(a)
        capi.acelib(a, out=host_out)
        t0 = time.perf_counter()
        for _ in range(5):
            capi.acelib(a, out=host_out)
        host_ms = 1e3 * (time.perf_counter() - t0) / 5
        log("acelib_ on host arrays (mixed): %.3f ms/call, %.3e atom-steps/s" % (host_ms, N / (1e-3 * host_ms)))

    # neighbour rebuild on the device (same pair set and order as the reference neilist)
    neighbors = importlib.import_module("magace_amd.neighbors")
    pos_t = T(s["pos"])
    mag_t = T(s["sdir"] * s["smag"][:, None])
    dn = neighbors.DeviceNeighbors([N], [1], [s["cell"]], 5.0)
    for _ in range(2):
        dn.build(pos_t, mag_t)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    nb_reps = 10
    for _ in range(nb_reps):
        dn.build(pos_t, mag_t)
    torch.cuda.synchronize()
    nb_ms = 1e3 * (time.perf_counter() - t0) / nb_reps
    assert dn.npairs == P, (dn.npairs, P)
    log("neighbour build: %.3f ms (%d pairs)" % (nb_ms, dn.npairs))

    o64, o32 = res["fp64"]["out"], res["mixed"]["out"]
    _, f64, m64, _ = systems.assemble(a, o64["eout"], o64["flist"], o64["tlist"], o64["tlist0"])
    _, f32, m32, _ = systems.assemble(a, o32["eout"], o32["flist"], o32["tlist"], o32["tlist0"])
    err = dict(energy_per_atom_max=float(np.abs(o32["eout"] - o64["eout"]).max()),
               force_max=float(np.abs(f32 - f64).max()), torque_max=float(np.abs(m32 - m64).max()),
               force_scale=float(np.abs(f64).max()), torque_scale=float(np.abs(m64).max()))
    log("mixed vs fp64:", err)

    raw = {2: info["raw2"], 3: info["raw3"], 4: info["raw4"]}
    fm = flops.flops_model(H, basis, raw, P / N)
    kernels = ("density", "adjoint", "forces")
    km = res["mixed"]["kernel_ms"]
    dom = int(np.argmax(km))
    ex = flops.executed(H, info["terms"], P / N)
    achieved = ex[kernels[dom]] * N / (km[dom] * 1e-3) / 1e12
    total_tf = fm["total"] * res["mixed"]["value"] / 1e12

    fitres = None
    if not args.no_md:
        fitres = fit_leg(pkg, td)
        log("fit (256 configurations):", {k: v for k, v in fitres.items() if k != "workload"})
    mdres = None
    if not args.no_md:
        mdres = md_leg(pkg, td)
        log("md (128000 atoms):", {k: v for k, v in mdres.items() if k != "workload"})

    cpu = orc = None
    if not args.no_cpu:
        try:
            cpu = cpu_baseline(pot, a, atoms_per_proc=min(args.cpu_sample, N // 16))
            log("cpu baseline:", cpu)
        except Exception as e:  # the headline line must still be printed
            log("cpu baseline failed:", e)
        try:
            orc = oracle_errors(pot, a, {"mixed": o32, "fp64": o64, "mixed_acc": res["mixed_acc"]["out"]},
                                min(2000, N))
            log("errors vs the oracle:", orc)
        except Exception as e:
            log("oracle comparison failed:", e)

    line = {
        "metric": "atom-steps/s E+F+torques, 16k Fe atoms: mixed vs FP64 @ force err <=1e-4 eV/A",
        "value": res["mixed"]["value"],
        "unit": "atom-steps/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": res["mixed"]["ms_per_step"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32+f64 (f32 splines/Y_lm/A/B products, f64 rho/energy/outputs)",
        "data": "synthetic (bcc Fe lattice, random coefficients from seed 2028)",
        "config": {"workload": "bcc Fe %dx%dx%d (%d atoms, %d pairs), cone spins <=30 deg, r_c 5.0 A, "
                               "header 10 3 2 6 / 7 1 6 1 / 3 1 3 1 (2043 B functions), E+F+dE/dm per step"
                               % (args.ncell, args.ncell, args.ncell, N, P),
                   "natoms": N, "pairs": P, "parallelism": "single GPU"},
        "fp64": {"value": res["fp64"]["value"], "ms_per_step": res["fp64"]["ms_per_step"],
                 "kernel_ms": res["fp64"]["kernel_ms"]},
        "mixed_over_fp64": res["mixed"]["value"] / res["fp64"]["value"],
        "mixed_acc": {"value": res["mixed_acc"]["value"], "ms_per_step": res["mixed_acc"]["ms_per_step"],
                      "kernel_ms": res["mixed_acc"]["kernel_ms"],
                      "note": "mixed with Kahan-compensated A sums and FP64 rho accumulation (MAGACE_MIXED_ACC)"},
        "mixed_error_vs_fp64": err,
        "kernel_ms": dict(zip(kernels, km)),
        "flops_per_atom_step": fm,
        "flops_executed_per_atom_step": ex,
        "achieved_tflops_total": total_tf,
        "roofline": {"bound": "valu", "kernel": kernels[dom], "achieved": achieved, "peak": PEAK["mixed"],
                     "unit": "TFLOP/s", "frac": achieved / PEAK["mixed"],
                     "note": "achieved counts the sums that the kernel executes (flops.executed), not the reference's "
                             "operations, of which it needs fewer; the vector units are also busy with what feeds them "
                             "(profiles/fe16k_lmax6_sq_counters.txt)",
                     "traffic": mixed_traffic(kernels[dom]) if args.ncell == 20 else None,
                     "traffic_unit": "bytes per launch (rocprofv3 FETCH_SIZE + WRITE_SIZE, copy-calibrated)"},
        "cpu_baseline": cpu,
        "error_vs_oracle": orc,
        "neighbor_build_ms": nb_ms,
        "acelib_host_arrays": None if host_ms is None else {
            "ms_per_call": host_ms, "atom_steps_per_s": N / (1e-3 * host_ms),
            "note": "acelib_ with host arrays, PCIe copies included (mixed)"},
        "spin_lattice_md": mdres,
        "batched_fit_step": fitres,
        "value_with_rebuild_every_10": N / (1e-3 * (res["mixed"]["ms_per_step"] + nb_ms / 10.0)),
    }
    if cpu:
        line["gpu_over_cpu"] = res["mixed"]["value"] / cpu["value"]
        line["gpu_over_cpu_single_core"] = res["mixed"]["value"] / cpu["single_core"]["value"]
    print(json.dumps(line))


if __name__ == "__main__":
    main()
