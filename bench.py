"""Throughput of one force evaluation (Moldy's eval_forces: make_sites,
force_calc, ewald and the glue) on one MI355X, inputs resident in HBM.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--precision mixed|fp64]

Workload: aqueous MgCl2, 32768 rigid 4-site waters + 600 Mg2+ + 1200 Cl-
(132,872 sites, 1.0 g/cm^3, r_c = 10 A, alpha = 0.30/A, k_c = 2.2302/A),
seeded synthetic configuration.  A step is one force evaluation; force-evals/s
equals MD steps/s and ns/day assumes dt = 1 fs.  Prints one JSON line.
"""
import argparse
import ctypes
import json
import math
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "force-evals/s + ns/day; mixed vs FP64 GPU at ≤1e-5 RMS rel force error"
DT_FS = 1.0

# Algorithmic work per (k-vector, site) in the reciprocal sum, counted on the
# reference loops (src/ewald.c:126-131, 528-531, 558-566): 6 flops for the
# q sin/cos addition step, 2 for the two sums, 9 for the force update.
FLOPS_SK_PER_KI = 8.0
FLOPS_FORCE_PER_KI = 9.0
# Real-space flops per evaluated pair (mk_r_sqr 11 + kernel LJ+erfc 39 +
# mk_forces 9), src/force.c:700-739, src/kernel.c:195-211.
FLOPS_PER_PAIR = 59.0
PEAK = {"fp64_vector": 78.6e12, "fp64_mfma": 78.6e12, "fp32_vector": 157.3e12, "fp16_mfma": 2.5e15}
# HBM bytes per dispatch (read + write) from rocprofv3 FETCH_SIZE/WRITE_SIZE
# passes on this workload, scaled by the counters' reading of a plain
# 512 MiB copy (profiles/saltwater132872_eval_forces_hbm_traffic.md).
MIB = float(1 << 20)
# One v_mfma_f32_16x16x32_f16 is 16384 flops.
MFMA_FLOPS = 16384.0
TRAFFIC_BYTES = {"ewald_mfma_force": (244.96 + 2.25) * MIB, "ewald_mfma_sk": (165.78 + 72.07) * MIB,
                 "ewald_sfac": (328.28 + 107.84) * MIB, "ewald_force": (1431.02 + 97.32) * MIB}


def build_workload(small=False):
    from moldy_amd import system
    if small:
        return system.salt_water(nwater=4096, nmg=75, ncl=150, seed=3)
    return system.salt_water(nwater=32768, nmg=600, ncl=1200, seed=3)


def rms_rel(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def time_gpu(eng, steps, warmup):
    import ctypes
    from moldy_amd import engine as E
    for _ in range(warmup):
        eng.eval_forces_device()
    eng.sync()
    eng.profile(True)
    t0 = time.perf_counter()
    for _ in range(steps):
        eng.eval_forces_device()
    eng.sync()
    t1 = time.perf_counter()
    prof = {}
    for name in ["binning", "realspace", "ewald_trig", "ewald_sfac", "ewald_kspace",
                 "ewald_force", "ewald_mfma_sk", "ewald_mfma_reduce", "ewald_mfma_force", "ewald_mfma_prep",
                 "ewald_grid_spread", "ewald_grid_forward", "ewald_grid_kspace", "ewald_grid_inverse",
                 "ewald_grid_gather", "make_sites", "glue"]:
        ms, n = eng.profile_get(name)
        if n:
            prof[name] = ms
    eng.profile(False)
    return (t1 - t0) / steps, prof


def mfma_issued(eng, ns):
    """MFMA flops the two mixed GEMMs issue per launch, from the engine's
    row plans (mgpu_mfma_plan): tiles multiply only the 16-wide l blocks
    their rows reach.
      back-projection: per 256-site block, 8 waves x per row tile 24 MFMAs
        (4 weight kinds x 2 site tiles x 3 hi/lo products) per l block;
      forward: per 32-site step of every site slice, 8 waves x 12 MFMAs
        (4 row tiles x 3 hi/lo products) per l block of the row tile.
    Also the counts with every tile over all NB blocks (no skipping)."""
    from moldy_amd import engine as E
    out = (ctypes.c_long * 4)()
    rc = E.lib().mgpu_mfma_plan(eng.h_, out)
    if rc:
        raise RuntimeError(f"mgpu_mfma_plan failed: {rc}")
    ftiles, fblocks, btiles, bblocks = list(out)
    nb = -(-(eng.last_info()[1].lmax + 1) // 16)
    nblk, steps = -(-ns // 256), -(-ns // 32)
    force = nblk * 8 * 24 * MFMA_FLOPS
    sk = steps * 8 * 12 * MFMA_FLOPS
    return dict(ewald_mfma_force=force * bblocks, ewald_mfma_sk=sk * fblocks,
                ewald_mfma_force_all_blocks=force * btiles * nb, ewald_mfma_sk_all_blocks=sk * ftiles * nb,
                forward_tiles=ftiles, forward_tile_blocks=fblocks, backprojection_tiles=btiles,
                backprojection_tile_blocks=bblocks, l_blocks=nb)


def mfma_rate(shape):
    """Sustained TFLOP/s of one FP16 MFMA shape on this device (16:
    16x16x32, 32: 32x32x16), from the library's probe."""
    import ctypes
    from moldy_amd import engine as E
    v = ctypes.c_double()
    rc = E.lib().mgpu_mfma_rate(0, shape, ctypes.byref(v))
    if rc:
        raise RuntimeError(f"mgpu_mfma_rate({shape}) failed: {rc}")
    return v.value


def pairlist_leg(eng, s, reps=5):
    """Link-cell binning and the reference's site neighbour lists (nab,
    pbctrans) for every cell, built on the GPU at the force cutoff; device
    time from HIP events on the engine stream, averaged over reps calls after
    one untimed call (which sizes the list buffers).  Algorithmic bytes:
    binning 32 B per site; lists 8 B per entry plus 8 B per cell."""
    eng.upload_state()
    eng.eval_forces_device()
    _, _, xyz, _ = eng.download()
    eng.pairlist(s.h, xyz)
    eng.profile(True)
    for _ in range(reps):
        out = eng.pairlist(s.h, xyz)
    t_bin, _ = eng.profile_get("binning")
    t_cnt, _ = eng.profile_get("pairlist_count")
    t_fill, _ = eng.profile_get("pairlist_fill")
    eng.profile(False)
    total = int(out["start"][-1])
    ncells = len(out["start"]) - 1
    list_bytes = 8.0 * total + 8.0 * ncells
    return dict(entries=total, cells=ncells, binning_ms=t_bin, count_ms=t_cnt, fill_ms=t_fill,
                binning_GBps=32.0 * s.nsites / (t_bin * 1e-3) / 1e9,
                list_fill_GBps=list_bytes / (t_fill * 1e-3) / 1e9,
                list_build_GBps=list_bytes / ((t_cnt + t_fill) * 1e-3) / 1e9)


def equilibrate(s, T=300.0, nblocks=8, nper=150, dt=0.001, precision=1, seed=7):
    """Relax the lattice start: short NVE blocks with the momenta rescaled to
    T after each (translational and rotational parts separately)."""
    from moldy_amd import engine as E, system, units
    e = E.ForceEngine(s, precision=precision)
    e.set_dynamics(system.Dynamics(step=dt))
    e.upload_state()
    mom, amom = s.thermal_momenta(T, seed=seed)
    e.upload_momenta(mom, amom)
    kT = units.KB * T
    for _ in range(nblocks):
        tr, _, _ = e.md_steps(nper, init_H_0=True)
        d = e.download_dynamics()
        kt, kr = tr[-1, 0], tr[-1, 1]
        ft = math.sqrt(1.5 * s.nmols * kT / kt)
        fr = math.sqrt(1.5 * s.nmols_r * kT / kr) if kr > 0 else 1.0
        e.upload_momenta(d["mom"] * ft, d["amom"] * fr)
    d = e.download_dynamics()
    e.close()
    return d


def nve_run(s, start, precision, nsteps, dt=0.001, chunk=250):
    """NVE from a common start: H = KE + PE at do_step's H_0 point per step,
    its linear drift and the rms deviation about the fit, and the device
    time per MD step (hipGraph-replayed steps, no host work between them)."""
    from moldy_amd import engine as E, system, units
    e = E.ForceEngine(s, precision=precision)
    e.set_dynamics(system.Dynamics(step=dt))
    e.upload_state(c_of_m=start["c_of_m"], quat=start["quat"])
    e.upload_momenta(start["mom"], start["amom"])
    e.md_steps(2, init_H_0=True)            # capture the graph outside the timing
    e.upload_state(c_of_m=start["c_of_m"], quat=start["quat"])
    e.upload_momenta(start["mom"], start["amom"])
    trs = []
    t0 = time.perf_counter()
    for c in range(nsteps // chunk):
        tr, _, _ = e.md_steps(chunk, init_H_0=(c == 0))
        trs.append(tr)
    t1 = time.perf_counter()
    e.close()
    tr = np.vstack(trs)
    H = tr[:, :4].sum(1) * units.CONV_E / s.nmols           # kJ/mol per molecule
    t_ps = np.arange(len(H)) * dt
    fit = np.polyfit(t_ps, H, 1)
    return dict(drift_kjmol_per_mol_per_ns=float(fit[0] * 1000.0),
                rms_fluct_kjmol_per_mol=float(np.std(H - np.polyval(fit, t_ps))),
                max_excursion_kjmol_per_mol=float(np.abs(H - H[0]).max()),
                ms_per_md_step=1e3 * (t1 - t0) / len(H), steps=len(H), dt_fs=dt * 1000)


def replica_leg(nrep, steps, seed=9):
    """64 rigid-water replicas of 256-2048 molecules (own box, alpha, r_c and
    k_c by Moldy's rule, own temperature 250-400 K), mixed precision, stepped
    together; schedule and launch shapes from the autotuner."""
    from moldy_amd import engine as E, system
    reps = system.water_replicas(nrep=nrep, seed=seed)
    engines = []
    for k, (s, T) in enumerate(reps):
        e = E.ForceEngine(s, precision=E.MIXED)
        e.set_dynamics(system.Dynamics(step=0.001))
        e.upload_state()
        e.upload_momenta(*s.thermal_momenta(T, seed=k))
        engines.append(e)
    b = E.Batch(engines)
    b.steps(2, init_H_0=True)
    sched, ms = b.autotune(trial_steps=8)
    b.steps(steps, init_H_0=True)              # buffers sized and steps captured outside the timing
    t0 = time.perf_counter()
    b.steps(steps)
    t1 = time.perf_counter()
    dt = (t1 - t0) / steps
    launches = None
    if sched == E.SCHED_GROUPED:
        g, own = b.grouped_plan()
        launches = dict(grouped_launches_per_step=g, replica_launches_per_step=own)
    sites = [s.nsites for s, _ in reps]
    b.close()
    for e in engines:
        e.close()
    return dict(replicas=nrep, total_sites=int(sum(sites)), min_sites=int(min(sites)),
                max_sites=int(max(sites)), schedule=E.SCHED_NAMES[sched],
                autotune_ms_per_step={E.SCHED_NAMES[i]: float(ms[i]) for i in range(len(ms))},
                ms_per_step=1e3 * dt, aggregate_force_evals_per_s=nrep / dt, launches=launches,
                per_replica_steps_per_s=1.0 / dt,
                per_replica_ns_per_day=86400.0 * 1e-6 * 1.0 / dt, dt_fs=1.0)


def cpu_model():
    """The host CPU's model name and the cores this process may use."""
    name = "unknown"
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                name = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    return name, len(os.sched_getaffinity(0))


def cpu_baseline(s):
    """The oracle (one core, strict IEEE) timed over one whole force
    evaluation of the same configuration: eval_forces with make_sites,
    force_calc over every pair and ewald over every k-vector."""
    from oracle.oracle import Oracle
    o = Oracle(s)
    xyz = o.make_sites()
    t0 = time.perf_counter()
    o.force_calc(xyz)
    t_real = time.perf_counter() - t0
    t0 = time.perf_counter()
    r = o.ewald(xyz)
    t_rec = time.perf_counter() - t0
    t_total = t_real + t_rec
    model, ncpu = cpu_model()
    return dict(value=1.0 / t_total, unit="force-evals/s", cores=1, kind="port",
                cpu=model, host_cores_available=ncpu,
                sample=(f"oracle/moldy_oracle.c, one whole evaluation of the same {s.nsites}-site "
                        f"configuration on one core of {model}: force_calc {t_real:.2f} s, ewald over all "
                        f"{r['info'].nhkl} k-vectors {t_rec:.2f} s"),
                seconds_per_eval=t_total)


def config_leg(name, s, dt_fs, precisions, reps=20, adjoint=False):
    """One configuration: force evaluations per second (inputs resident,
    launch shapes autotuned) and MD steps per second (hipGraph-replayed
    do_steps) at each precision; for the silica, the parameter adjoint
    (dE/dtheta and the force cotangent product) per second."""
    from moldy_amd import engine as E, system
    out = dict(workload=name, sites=s.nsites)
    for p in precisions:
        e = E.ForceEngine(s, precision=p)
        e.upload_state()
        if s.control.alpha > 0:
            e.autotune()
        t, _ = time_gpu(e, reps, 2)
        key = "fp64" if p == E.FP64 else "mixed"
        out[f"{key}_evals_per_s"] = 1.0 / t
        out[f"{key}_ms_per_eval"] = 1e3 * t
        e.set_dynamics(system.Dynamics(step=dt_fs * 1e-3))
        e.upload_state()
        e.upload_momenta(*s.thermal_momenta(300.0 if s.nmols_r else 120.0, seed=2))
        e.md_steps(2, init_H_0=True)
        e.sync()
        t0 = time.perf_counter()
        e.md_steps(reps)
        e.sync()
        tm = (time.perf_counter() - t0) / reps
        out[f"{key}_md_steps_per_s"] = 1.0 / tm
        out[f"{key}_md_ns_per_day"] = 86400.0 * 1e-6 * dt_fs / tm
        if adjoint and p == E.FP64:
            e.upload_state()
            e.eval_forces_device()
            v = np.random.default_rng(0).standard_normal((3, s.nsites))
            e.adjoint(v=v)
            e.sync()
            t0 = time.perf_counter()
            for _ in range(5):
                e.adjoint(v=v)
            e.sync()
            ta = (time.perf_counter() - t0) / 5
            out["fp64_adjoint_per_s"] = 1.0 / ta
            out["fp64_adjoint_ms"] = 1e3 * ta
            out["adjoint_parameters"] = e.theta_count()
        e.close()
    out["dt_fs"] = dt_fs
    return out


def nve_drift(s, starts=3, nsteps=20000, dt=0.0005):
    """NVE drift of H = KE + PE per molecule, FP64 and mixed, from several
    independently equilibrated starts (the same starts for both precisions):
    the linear drift per ns of each run, their mean and spread, and the rms
    fluctuation about the fit."""
    from moldy_amd import engine as E
    out = {}
    starts_state = [equilibrate(s, seed=7 + k) for k in range(starts)]
    for name, p in (("fp64", E.FP64), ("mixed", E.MIXED)):
        runs = [nve_run(s, st, p, nsteps, dt=dt, chunk=500) for st in starts_state]
        d = np.array([r["drift_kjmol_per_mol_per_ns"] for r in runs])
        out[name] = dict(drift_kjmol_per_mol_per_ns=[float(x) for x in d],
                         drift_mean=float(d.mean()), drift_sd=float(d.std(ddof=1)) if len(d) > 1 else 0.0,
                         abs_drift_mean=float(np.abs(d).mean()),
                         rms_fluct_kjmol_per_mol=float(np.mean([r["rms_fluct_kjmol_per_mol"] for r in runs])),
                         ms_per_md_step=float(np.mean([r["ms_per_md_step"] for r in runs])))
        print(f"[bench] nve {name}: {out[name]}", file=sys.stderr, flush=True)
    out.update(workload=f"rigid 4-site water, {s.nmols} molecules ({s.nsites} sites), r_c "
                        f"{s.control.cutoff} A, alpha {s.control.alpha}/A",
               starts=starts, steps_per_run=nsteps, dt_fs=dt * 1000,
               start="8 x 150 steps at 1 fs with momenta rescaled to 300 K after each block, "
                     "one seed per start")
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--precision", choices=["mixed", "fp64"], default="mixed")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--small", action="store_true", help="17k-site variant (smoke only)")
    ap.add_argument("--mixed-only", action="store_true",
                    help="profiling runs: skip the FP64 leg and the error comparison")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="only run a plain 512 MiB device copy (the PMC byte-count reference)")
    ap.add_argument("--replicas", type=int, default=64,
                    help="replicas in the batched leg (0: skip)")
    ap.add_argument("--nve-steps", type=int, default=20000,
                    help="NVE steps per start and precision for the drift comparison (0: skip)")
    ap.add_argument("--nve-dt-fs", type=float, default=0.5,
                    help="NVE time step in fs (0.5: the step of the reference's TIP4P example)")
    ap.add_argument("--nve-starts", type=int, default=3, help="independent starts for the NVE drift")
    ap.add_argument("--no-configs", dest="configs", action="store_false",
                    help="skip the legs of configurations 1, 2 and 4")
    a = ap.parse_args()
    if a.gpus != 1:
        print(f"bench.py measures one GPU; --gpus {a.gpus} is not supported (the force "
              "path is built for a single MI355X and runs on one GPU only)",
              file=sys.stderr)
        sys.exit(2)
    if a.copy_calibration:
        import torch
        x = torch.ones(128 << 20, dtype=torch.float32, device="cuda")
        y = torch.empty_like(x)
        for _ in range(3):
            y.copy_(x)
        torch.cuda.synchronize()
        print(json.dumps(dict(copy_bytes_read=x.numel() * 4, copy_bytes_written=y.numel() * 4)))
        return
    from moldy_amd import engine as E
    s = build_workload(a.small)
    print(f"[bench] workload {s.name}: {s.nsites} sites", file=sys.stderr, flush=True)
    eng = E.ForceEngine(s, precision=E.FP64)
    eng.upload_state()

    if a.mixed_only:
        eng.set_precision(E.MIXED)
        eng.autotune()
        tmx, profmx = time_gpu(eng, a.steps, a.warmup)
        print(json.dumps(dict(ms_per_eval=1e3 * tmx, kernel_ms=profmx)))
        return
    # FP64 leg (launch shapes from the autotuner)
    tuned = {"fp64": eng.autotune()}
    t64, prof64 = time_gpu(eng, a.steps, a.warmup)
    fc, ew = eng.last_info()
    pe64, _, st64 = eng.eval_forces_device()
    f64, tq64, _, sf64 = eng.download()
    print(f"[bench] fp64 {1e3 * t64:.3f} ms/eval {prof64}", file=sys.stderr, flush=True)
    nk, ns = ew.nhkl, s.nsites

    res = dict(metric=METRIC, n_gpus=1, steps=a.steps, warmup=a.warmup,
               higher_is_better=True, scaling="weak", vs_baseline=None, data="synthetic")
    mixed = None
    if a.precision == "mixed":
        eng.set_precision(E.MIXED)
        tuned["mixed"] = eng.autotune()
        tmx, profmx = time_gpu(eng, a.steps, a.warmup)
        pemx, _, stmx = eng.eval_forces_device()
        fmx, tqmx, _, sfmx = eng.download()
        if "ewald_mfma_force" in profmx:   # the direct reciprocal sum (small systems, frameworks)
            res["mfma_issued_per_launch"] = mfma_issued(eng, s.nsites)
        print(f"[bench] mixed {1e3 * tmx:.3f} ms/eval {profmx}", file=sys.stderr, flush=True)
        mixed = dict(t=tmx, prof=profmx,
                     err=dict(site_force=rms_rel(sfmx, sf64), mol_force=rms_rel(fmx, f64),
                              torque=rms_rel(tqmx, tq64) if s.nmols_r else 0.0,
                              pe_real=abs(pemx[0] - pe64[0]) / abs(pe64[0]),
                              pe_recip=abs(pemx[1] - pe64[1]) / abs(pe64[1]),
                              stress=rms_rel(stmx, st64)))
    t = mixed["t"] if mixed else t64
    evals = 1.0 / t
    res.update(value=evals, unit="force-evals/s", ms_per_step=1e3 * t,
               ns_per_day=evals * DT_FS * 86400 / 1e6,
               dtype=("f64" if not mixed else
                      "f32 pairs + f16x2 MFMA Ewald + f64 reductions" if "ewald_mfma_force" in mixed["prof"] else
                      "f32 pairs + f32 gridded Ewald with f64 transforms + f64 reductions"),
               config=dict(workload=f"aqueous MgCl2: 32768 rigid 4-site water + 600 Mg2+ + 1200 Cl- "
                                    f"({ns} sites)", sites=ns, k_vectors=nk, cutoff_A=10.0,
                           alpha_per_A=0.30, k_cutoff_per_A=round(s.control.k_cutoff, 4),
                           cells=[fc.nx, fc.ny, fc.nz], dt_fs=DT_FS,
                           precision=a.precision))
    # launch shapes of the direct reciprocal sum (the gridded sum has none)
    shapes = {}
    if "ewald_force" in prof64:
        shapes["fp64"] = dict(fp64_backprojection_parts=tuned["fp64"][1])
    if mixed and "ewald_mfma_force" in mixed["prof"]:
        shapes["mixed"] = dict(sk_workgroups=tuned["mixed"][0], backprojection_rounds=tuned["mixed"][1])
    if shapes:
        res["autotuned_shapes"] = shapes
    res["fp64_evals_per_s"] = 1.0 / t64
    res["fp64_ms_per_eval"] = 1e3 * t64
    if mixed:
        res["mixed_over_fp64"] = t64 / mixed["t"]
        res["mixed_error_vs_fp64"] = mixed["err"]
    prof = mixed["prof"] if mixed else prof64
    # roofline of the dominant kernel: with the direct reciprocal sum its
    # back-projection, the longest kernel that runs alone; with the gridded
    # sum the real-space pass (timed while it shares the GPU with the
    # reciprocal stages when the two streams overlap)
    dom = next(k for k in ("ewald_mfma_force", "ewald_force", "realspace") if k in prof)
    pairs = 0.5 * ns * ns / s.volume() * 4.0 / 3.0 * np.pi * s.control.cutoff ** 3
    kind = {"realspace": ("fp32_vector" if mixed else "fp64_vector", FLOPS_PER_PAIR * pairs),
            "ewald_sfac": ("fp64_mfma", FLOPS_SK_PER_KI * nk * ns),
            "ewald_force": ("fp64_vector", FLOPS_FORCE_PER_KI * nk * ns),
            "ewald_mfma_sk": ("fp16_mfma", FLOPS_SK_PER_KI * nk * ns),
            "ewald_mfma_force": ("fp16_mfma", FLOPS_FORCE_PER_KI * nk * ns)}.get(dom)
    if kind:
        peak = PEAK[kind[0]]
        ach = kind[1] / (prof[dom] * 1e-3)
        res["roofline"] = dict(kernel=dom, bound="mfma" if "mfma" in kind[0] else "valu",
                               achieved=ach / 1e12, peak=peak / 1e12, unit="TFLOP/s",
                               frac=ach / peak, traffic=TRAFFIC_BYTES.get(dom),
                               flops_per_launch=kind[1], avg_ms=prof[dom])
        if dom in res.get("mfma_issued_per_launch", {}):
            # the matrix-core work the kernel issues, beside the rate its
            # instruction sustains on this device (the published dense peak
            # assumes the faster 32x32x16 shape)
            issued = res["mfma_issued_per_launch"][dom] / (prof[dom] * 1e-3)
            r16, r32 = mfma_rate(16), mfma_rate(32)
            res["roofline"].update(instruction="v_mfma_f32_16x16x32_f16", issued=issued / 1e12,
                                   instruction_peak=r16, issued_frac_of_instruction_peak=issued / 1e12 / r16,
                                   mfma_32x32x16_peak=r32)
    res["kernel_ms"] = prof
    res["pairlist"] = pairlist_leg(eng, s)
    print(f"[bench] pairlist: {res['pairlist']}", file=sys.stderr, flush=True)
    eng.close()
    if a.configs:
        from moldy_amd import system
        legs = {}
        legs["config1_argon"] = config_leg("864 LJ argon, fcc 6x6x6, r_c 10.2 A", system.argon_fcc(ncell=6),
                                           10.0, (E.FP64,))
        legs["config2_water"] = config_leg("4096 rigid 4-site water, alpha 0.30, r_c 9 A",
                                           system.water_box(4096, seed=1), 1.0, (E.FP64, E.MIXED))
        legs["config4_silica"] = config_leg("8000 Si + 16000 O, Buckingham + Ewald, r_c 10 A",
                                            system.silica(ncell=10, seed=7), 1.0, (E.FP64,), adjoint=True)
        for k, v in legs.items():
            print(f"[bench] {k}: {v}", file=sys.stderr, flush=True)
        res["configs"] = legs
    if a.nve_steps > 0:
        from moldy_amd import system
        res["nve"] = nve_drift(system.water_box(4096, seed=1), starts=a.nve_starts, nsteps=a.nve_steps,
                               dt=a.nve_dt_fs * 1e-3)
        res["md_ns_per_day_nve_water"] = {
            k: 86400.0 * a.nve_dt_fs * 1e-6 / (res["nve"][k]["ms_per_md_step"] * 1e-3) for k in ("fp64", "mixed")}
    if a.replicas > 0:
        res["replica_batch"] = replica_leg(a.replicas, max(a.steps, 30))
        print(f"[bench] replicas: {res['replica_batch']}", file=sys.stderr, flush=True)
    if not a.no_cpu:
        cb = cpu_baseline(s)
        res["cpu_baseline"] = cb
    print(json.dumps(res))


if __name__ == "__main__":
    main()
