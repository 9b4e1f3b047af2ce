"""Benchmark of the MPDATA advection step on one MI355X.

Headline workload (the largest configuration that fits one GPU): one
4096 x 4096 x 50 domain (839 M cells, dx 250 m, fractal terrain with a
3000 m ridge line, a 20 m/s jet at 8 km plus a terrain-forced perturbation,
w from continuity, dt at Courant 0.5), 12 species (qv, theta, qc, qr, qs,
qi, qg, ni, nr, ns, ng and a passive tracer), mpdata_order 2 with FCT,
advect_density on.  A step is one advect() call (Courant numbers plus every
species through all MPDATA passes) with all inputs resident in HBM.
value = cell-species updates per second = nx*ny*nz*species*steps / t.

Variants on that domain:
  batched_mixed  fused species-batched kernels, qv and theta FP32 and the
                 ten others stored in BF16 with power-of-two scaling and
                 stochastic rounding (the value reported);
  batched        the same kernels with every species FP32 (bit-identical to
                 the FP32 oracle);
  plain          one kernel per MPDATA pass and species, every species FP32:
                 the drop-in form the mixed variant is compared with.
The CPU baseline is the FP32 oracle (a scalar C restatement of the
reference) on the host cores, one subdomain per core as ICAR runs its
images, on a strip of the same domain.

Beside it (unless --no-extras): the 1024 x 1024 x 30, 10-species domain at
mpdata_order 3 + FCT in its three variants, a launch-bound 256x64x20 case
eager and from a HIP graph, the 48-domain ensemble, the standard scheme,
the host hand-off and the kernels next to advect.

Prints one JSON line.  Options: --steps K --warmup W --gpus N (1 only)
--workload c5|c2 (c2 puts the 1024x1024x30 domain in the headline line)
--no-cpu --no-extras --no-plain, and for the c2 extras --no-small
--no-ensemble --no-std --no-handoff --no-wind.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK = 8.0e12  # B/s, MI355X HBM3E
# wave64 VALU instructions per second: 256 CUs x 4 SIMDs x 2.4 GHz, 4 cycles each
VALU_ISSUE_PEAK = 256 * 4 * 2.4e9 / 4


def log(msg: str) -> None:
    print(msg, file=sys.stderr, flush=True)


def measure(case, variant: int, steps: int, warmup: int, profile: bool = True,
            graph: bool = False):
    from hicar_amd.advection import MpdataAdvection
    case.options.kernel_variant = variant
    st = MpdataAdvection(case.domain, case.options)
    try:
        st.set_graph(graph)
        def loop(n):
            if graph:
                st.run(case.dt, n)
            else:  # a step is one advect() call (run() forms the Courant numbers once)
                for _ in range(n):
                    st.advect(case.dt)

        loop(warmup)
        st.sync()
        if graph:  # record the timed loop once so that the timed call replays it
            loop(steps)
            st.sync()
        st.profile(profile)
        t0 = time.perf_counter()
        loop(steps)
        st.sync()
        t1 = time.perf_counter()
        stats = st.kernel_stats() if profile else {}
        st.profile(False)
        cfg = st.launch_config()
    finally:
        st.close()
    if profile:
        stats["_launch_config"] = {"corr_cfg": cfg[0], "column_chunks": cfg[1]}
    return t1 - t0, stats


def measure_ensemble(steps: int, warmup: int, n: int = 48):
    """The ensemble workload: n independent domains (nx, ny ~ U[64,512], nz in
    {20,30,40}, 6 FP32 species each, order 2 + FCT), advanced by one launch
    per pass over all of them, each with its own dt; the step loop is
    replayed from a HIP graph (and, for comparison, run eagerly)."""
    import numpy as np

    from hicar_amd import synthetic
    from hicar_amd.advection import Ensemble, MpdataAdvection
    t0 = time.perf_counter()
    cases = synthetic.config3(n, steps=steps)
    gen_s = time.perf_counter() - t0
    members = [MpdataAdvection(c.domain, c.options) for c in cases]
    ens = Ensemble(members)
    dts = np.array([c.dt for c in cases], np.float32)
    cs = sum(c.domain.nx * c.domain.ny * c.domain.nz * len(c.domain.species) for c in cases)
    out = {"domains": n, "cells": sum(c.domain.nx * c.domain.ny * c.domain.nz for c in cases),
           "species": len(cases[0].domain.species), "mpdata_order": 2, "fct": True,
           "generation_s": gen_s}
    try:
        for graph in (False, True):
            ens.run(dts, warmup, 1, 2, graph=graph)
            ens.sync()
            if graph:  # record the timed loop once; the timed call replays it
                ens.run(dts, steps, 1, 2, graph=True)
                ens.sync()
            t0 = time.perf_counter()
            ens.run(dts, steps, 1, 2, graph=graph)
            ens.sync()
            t = time.perf_counter() - t0
            out["graph" if graph else "eager"] = {"value": cs * steps / t,
                                                  "ms_per_step": 1e3 * t / steps}
        out["launch_config"] = dict(zip(("corr_cfg", "column_chunks"), ens.launch_config()))
    finally:
        ens.close()
        for m in members:
            m.close()
    return out


def measure_std(nx: int, ny: int, steps: int, warmup: int):
    """The standard scheme (adv=1) on the same 1024x1024x30, 10-species
    domain with the settings of run/complete_icar_options.nml: h_order 5,
    v_order 3, the WRF monotonic limiter and RK3, Courant 1.2 (w balances the
    scheme's mass fluxes).  A step is one advect(): the mass fluxes, then per
    species three RK3 stages, the last one limited."""
    from hicar_amd import synthetic
    case = synthetic.config_std(nx=nx, ny=ny)
    d = case.domain
    S = len(d.species)
    t, stats = measure(case, 0, steps, warmup)
    stats.pop("_launch_config", None)
    cells = d.nx * d.ny * d.nz
    return {"value": cells * S * steps / t, "unit": "cell-species updates/s",
            "ms_per_step": 1e3 * t / steps, "species": S, "h_order": 5, "v_order": 3,
            "flux_corr": 1, "rk3": True, "dt": case.dt,
            "parity": "bit-identical to the FP32 oracle",
            "kernels": {k: {"avg_ms": v["total_ms"] / v["launches"], "launches": v["launches"],
                            "achieved_GBps": v["alg_bytes"] / v["total_ms"] / 1e6}
                        for k, v in stats.items()}}


def measure_host_handoff(case, steps: int, warmup: int):
    """What keeping ICAR's CPU physics in the loop costs the step: the
    species' upload and download (the minimal policy uploads what the CPU
    physics changed, all species after mp, and downloads what advect
    changed, all species, every step), and what an output snapshot every
    step adds to the step (its copy out overlaps the following steps)."""
    from hicar_amd.advection import MpdataAdvection
    d = case.domain
    nbytes = 4.0 * d.nx * d.ny * d.nz * len(d.species)
    case.options.kernel_variant = 1
    saved = dict(d.storage)
    d.storage.clear()  # FP32 species, as the host holds them
    st = MpdataAdvection(d, case.options)
    out = {}
    try:
        st.run(case.dt, warmup)
        st.sync()
        t0 = time.perf_counter()
        for _ in range(3):
            st.upload(fields=False, species=True)
        t1 = time.perf_counter()
        for _ in range(3):
            st.download(species=True)
        t2 = time.perf_counter()
        up, down = (t1 - t0) / 3, (t2 - t1) / 3
        out["species_bytes"] = nbytes
        out["upload_ms"] = 1e3 * up
        out["download_ms"] = 1e3 * down
        out["upload_GBps"] = nbytes / up / 1e9
        out["download_GBps"] = nbytes / down / 1e9
        t0 = time.perf_counter()
        st.run(case.dt, steps)
        st.sync()
        plain = (time.perf_counter() - t0) / steps
        # one snapshot of every species, then the steps while it is copied out
        # (a first one allocates and pins the staging)
        st.snapshot(species=True)
        st.snapshot_wait()
        t0 = time.perf_counter()
        st.snapshot(species=True)
        st.run(case.dt, steps)
        st.sync()
        t1 = time.perf_counter()
        st.snapshot_wait()
        t2 = time.perf_counter()
        out["step_ms"] = 1e3 * plain
        out["step_ms_while_snapshot_in_flight"] = 1e3 * (t1 - t0) / steps
        out["snapshot_to_host_ms"] = 1e3 * (t2 - t0)
    finally:
        st.close()
        d.storage.update(saved)
    return out


def measure_wind_steps(case, reps: int = 10):
    """The steps next to advect on the device copies: balance_uvw and
    compute_dt on the workload's winds, and apply_forcing of every species
    with the one-image relaxation filter: HIP-event time per launch and
    algorithmic GB/s (inputs read once, outputs written once)."""
    import numpy as np

    from hicar_amd import synthetic
    from hicar_amd.advection import MpdataAdvection
    case.options.kernel_variant = 1
    st = MpdataAdvection(case.domain, case.options)
    out = {}
    try:
        dzl = synthetic.dz_levels(case.domain.nz).astype(np.float32)
        st.set_relax_filter(True, True, True, True, halo=2)
        zero = np.zeros(case.domain.shape, np.float32)
        for n in st.names:
            if case.domain.storage.get(n, (0, 0))[0] == 0:
                st.set_forcing(n, case.domain.species[n], zero)
        st.balance_w()
        st.compute_dt(0.9, 3, dzl)
        st.apply_forcing(10.0)
        st.sync()
        st.profile(True)
        for _ in range(reps):
            st.balance_w()
            st.compute_dt(0.9, 3, dzl)
            st.apply_forcing(10.0)
        stats = st.kernel_stats()
        st.profile(False)
        for name in ("wind_balance", "dt_bound", "forcing"):
            k = stats[name]
            ms = k["total_ms"] / k["launches"]
            gbs = k["alg_bytes"] / k["total_ms"] / 1e6
            out[name] = {"avg_ms": ms, "achieved_GBps": gbs, "hbm_frac": gbs * 1e9 / HBM_PEAK}
    finally:
        st.close()
    return out


def set_bf16(case):
    from hicar_amd import _lib, synthetic
    d = case.domain
    for n, a in d.species.items():
        if n not in ("qv", "theta"):
            d.storage[n] = (_lib.STORE_BF16_SR, synthetic.pow2_scale(a, _lib.STORE_BF16_SR))


# profiler kernel names of the timed kernels
KERNEL_SYMBOL = {"fused_corrective_pass": "k_corr", "fused_first_pass": "k_first",
                 "face_coefficients": "k_coef", "courant": "k_courant", "upwind": "k_upwind",
                 "pseudo_velocity": "k_pseudo", "fct": "k_fct", "copy": "k_copy"}


def _traffic_file(workload: str) -> str:
    return os.path.join(ROOT, "profiles", f"traffic_{workload}.txt")


def read_traffic(kernel: str, workload: str = "c2_1024x1024x30"):
    """HBM bytes per launch of a kernel from the committed PMC summary of the
    workload (profiles/traffic_<workload>.txt: lines 'kernel fetch_bytes
    write_bytes')."""
    path = _traffic_file(workload)
    if os.path.exists(path):
        for line in open(path):
            parts = line.split()
            if len(parts) == 3 and parts[0] == kernel:
                try:
                    return float(parts[1]) + float(parts[2])
                except ValueError:
                    pass
    return None


def step_bytes(d) -> float:
    """Compulsory HBM bytes of one step: the nine input fields read once and
    every species read and written once at its storage width,
    4*(5*N + 2*N_u + 2*N_v) + sum_s 2*b_s*N."""
    from hicar_amd import _lib
    N = d.nx * d.ny * d.nz
    Nu = (d.nx + 1) * d.nz * d.ny
    Nv = d.nx * d.nz * (d.ny + 1)
    b = 4 * (5 * N + 2 * Nu + 2 * Nv)
    for n in d.species:
        st = d.storage.get(n, (_lib.STORE_F32, 0))[0]
        b += 2 * (4 if st == _lib.STORE_F32 else 2) * N
    return float(b)


def read_valu(kernel: str, workload: str = "c2_1024x1024x30"):
    """VALU wave-instructions per launch of a kernel from the committed PMC
    summary of the workload (lines 'valu kernel count')."""
    path = _traffic_file(workload)
    if os.path.exists(path):
        for line in open(path):
            parts = line.split()
            if len(parts) == 3 and parts[0] == "valu" and parts[1] == kernel:
                return float(parts[2])
    return None


def host_cores() -> dict:
    """Threads this process may use (its CPU affinity, the host's share for
    one GPU) and the host's own counts (logical CPUs, physical cores as lscpu
    lists them)."""
    import subprocess
    try:
        share = len(os.sched_getaffinity(0))
    except AttributeError:
        share = os.cpu_count() or 1
    phys = None
    try:
        r = subprocess.run(["lscpu", "-p=CORE,SOCKET"], capture_output=True, text=True, timeout=10)
        cores = {ln for ln in r.stdout.splitlines() if ln and not ln.startswith("#")}
        phys = len(cores) or None
    except (OSError, subprocess.SubprocessError):
        pass
    return {"threads": max(1, min(16, share)), "logical_cpus": os.cpu_count(),
            "physical_cores": phys}


def _image(d, j0: int, j1: int):
    """Rows j0..j1-1 of the domain as a subdomain of its own (an ICAR image:
    its outer ring, here the rows next to its neighbours, is its halo)."""
    from hicar_amd.domain import Domain
    sub = Domain(d.nx, j1 - j0, d.nz, d.dx, halo=d.halo)
    for n in d.FIELDS:
        rows = j1 - j0 + (1 if n in ("v", "jacobian_v") else 0)
        getattr(sub, n)[...] = getattr(d, n)[j0:j0 + rows]
    return sub, {n: a[j0:j1].copy() for n, a in d.species.items()}


def cpu_baseline(case, rows: int = None):
    """The FP32 oracle (a scalar C restatement of the reference) on the host
    cores, parallel the way ICAR is: one image per core
    (src/objects/grid_obj.f90:40 decomposes the domain; between halo
    exchanges the images advance independently).  The sample is the strip
    of the first `rows` rows (all of them by default) cut into one image of
    rows/threads owned rows per thread, each with the MPDATA halo of 2 rows
    on its inner sides; one advect() of every species on every image,
    timed around the parallel map (ctypes releases the GIL, so the C code
    runs in parallel).  The rate counts owned cells.  For reference, one
    image alone on one thread."""
    from concurrent.futures import ThreadPoolExecutor

    import numpy as np

    from oracle.oracle import Oracle
    orc = Oracle(np.float32)
    d = case.domain
    S = len(d.species)
    hc = host_cores()
    threads = hc["threads"]
    rows = min(rows or d.ny, d.ny)
    per = max(3, rows // threads)
    images = []
    for j0 in range(0, rows - per + 1, per):
        a, b = max(0, j0 - 2), min(d.ny, j0 + per + 2)
        images.append(_image(d, a, b) + (per,))
    owned = sum(p for _, _, p in images) * d.nx * d.nz * S

    def one(img):
        sub, sp, _ = img
        orc.advect(sub, case.options, case.dt, species=sp)

    with ThreadPoolExecutor(threads) as ex:
        list(ex.map(one, images[:1]))  # warm the oracle's code and pages once
        t0 = time.perf_counter()
        list(ex.map(one, images))
        t = time.perf_counter() - t0
    t1 = time.perf_counter()
    one(images[0])
    t1 = time.perf_counter() - t1
    n1 = images[0][2] * d.nx * d.nz * S
    return {"value": owned / t, "unit": "cell-species updates/s", "cores": threads,
            "kind": "port", "host": hc,
            "sample": f"one advect() of {S} species on rows 0..{rows - 1} of the "
                      f"{d.nx}x{d.ny}x{d.nz} domain, as {len(images)} images of {per} owned "
                      f"rows (+2 halo rows inside), one per thread on {threads} threads "
                      f"({t:.1f} s)",
            "single_thread": {"value": n1 / t1, "cores": 1,
                              "sample": f"one of those images on one thread ({t1:.1f} s)"}}


def kernel_table(stats) -> dict:
    return {k: {"avg_ms": v["total_ms"] / v["launches"], "launches": v["launches"],
                "achieved_GBps": v["alg_bytes"] / v["total_ms"] / 1e6}
            for k, v in stats.items()}


def roofline_of(stats, d, units_per_launch, workload: str, kernel: str) -> dict:
    """The HBM roofline of one kernel: the step's compulsory bytes per
    cell-species times the cell-species one launch advances, over the live
    HIP-event launch duration; traffic and VALU count from the committed PMC
    summary of the workload."""
    S = len(d.species)
    cells = d.nx * d.ny * d.nz
    per_unit = step_bytes(d) / (cells * S)
    ks = stats[kernel]
    avg_s = ks["total_ms"] / ks["launches"] / 1e3
    achieved = per_unit * units_per_launch / avg_s
    sym = KERNEL_SYMBOL.get(kernel, kernel)
    out = {"bound": "hbm", "achieved": achieved / 1e9, "peak": HBM_PEAK / 1e9, "unit": "GB/s",
           "frac": achieved / HBM_PEAK, "traffic": read_traffic(sym, workload), "kernel": kernel,
           "avg_launch_ms": avg_s * 1e3, "bytes_per_cell_species": per_unit,
           "cell_species_per_launch": units_per_launch,
           "kernel_own_bytes_per_launch": ks["alg_bytes"] / ks["launches"]}
    vi = read_valu(sym, workload)
    if vi is not None:
        out["valu"] = {"wave_instr_per_launch": vi, "achieved": vi / avg_s / 1e9,
                       "peak": VALU_ISSUE_PEAK / 1e9, "unit": "G wave-instr/s",
                       "frac": vi / avg_s / VALU_ISSUE_PEAK,
                       "lane_instr_per_cell_species": 64.0 * vi / units_per_launch}
    return out


def c5_line(args) -> dict:
    """The headline: the 4096x4096x50 domain, 12 species, order 2 + FCT, in
    its three variants (batched_mixed is the value), and the CPU baseline on
    a strip of the same domain."""
    from hicar_amd import _lib, synthetic
    t0 = time.perf_counter()
    case = synthetic.config5(steps=args.steps, log=log)
    gen_s = time.perf_counter() - t0
    d = case.domain
    S = len(d.species)
    cells = d.nx * d.ny * d.nz
    mixed = dict(d.storage)
    log(f"4096x4096x50 domain generated in {gen_s:.0f} s")
    todo = ["batched_mixed", "batched"] + ([] if args.no_plain else ["plain"])
    results = {}
    for name in todo:
        d.storage.clear()
        if name == "batched_mixed":
            d.storage.update(mixed)
        log(f"variant {name}: {args.warmup} warmup + {args.steps} timed steps ...")
        try:
            t, stats = measure(case, 0 if name == "plain" else 1, args.steps, args.warmup)
        except _lib.IcarAdvError as e:  # e.g. a variant that does not fit in memory
            log(f"  {name}: not measured ({e})")
            results[name] = {"error": str(e)}
            continue
        lc = stats.pop("_launch_config", None)
        results[name] = {"seconds": t, "value": cells * S * args.steps / t, "stats": stats,
                         "b_step": step_bytes(d), "launch_config": lc}
        log(f"  {name}: {results[name]['value'] / 1e9:.2f} G cell-species/s, "
            f"{1e3 * t / args.steps:.1f} ms/step")
    d.storage.clear()
    d.storage.update(mixed)
    r = results["batched_mixed"]
    roof = roofline_of(r["stats"], d, cells * S, "c5_4096x4096x50", "fused_corrective_pass")
    variants = {}
    for k, v in results.items():
        if "error" in v:
            variants[k] = v
            continue
        variants[k] = {"value": v["value"], "ms_per_step": 1e3 * v["seconds"] / args.steps,
                       "compulsory_hbm_fraction": v["b_step"] * args.steps / v["seconds"] / HBM_PEAK,
                       "bytes_per_cell_species": v["b_step"] / (cells * S),
                       "launch_config": v["launch_config"] if k != "plain" else None,
                       "kernels": kernel_table(v["stats"])}
    out = {
        "metric": "MPDATA cell-species updates/s & % HBM roofline, plain FP32 vs batched/mixed",
        "value": r["value"], "unit": "cell-species updates/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": 1e3 * r["seconds"] / args.steps, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "storage": {n: ("f32" if n not in d.storage else _lib.STORE_NAMES[d.storage[n][0]])
                    for n in d.species},
        "parity": "batched and plain bit-identical to the FP32 oracle; batched_mixed equal to the "
                  "FP32 oracle stepped on the 16-bit values with one rounding per step",
        "config": {"workload": f"single domain {d.nx}x{d.ny}x{d.nz}, {S} species (qv, theta FP32; "
                               "ten BF16 with power-of-two scaling and stochastic rounding), "
                               "mpdata_order 2 + FCT, advect_density, Courant 0.5",
                   "nx": d.nx, "ny": d.ny, "nz": d.nz, "species": S, "mpdata_order": 2,
                   "fct": True, "variant": "batched_mixed", "dt": case.dt,
                   "generation_s": gen_s, "variants_run": todo},
        "roofline": roof,
        "compulsory_hbm_fraction": r["b_step"] * args.steps / r["seconds"] / HBM_PEAK,
        "variants": variants,
    }
    if "value" in results.get("plain", {}):
        out["mixed_vs_plain"] = r["value"] / results["plain"]["value"]
    if "value" in results.get("batched", {}):
        out["mixed_vs_batched_fp32"] = r["value"] / results["batched"]["value"]
    if not args.no_cpu:
        log("CPU baseline (oracle, one image per thread on a 512-row strip) ...")
        out["cpu_baseline"] = cpu_baseline(case, rows=512)
    return out


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--workload", choices=("c5", "c2"), default="c5",
                    help="c5: the 4096x4096x50 domain, 12 species, mixed precision (the "
                         "headline); c2: the 1024x1024x30, 10-species domain in the headline line")
    ap.add_argument("--variant", choices=("plain", "batched", "batched_bf16", "all"),
                    default="all", help="variants of the c2 domain")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    ap.add_argument("--no-plain", action="store_true",
                    help="skip the plain variant of the 4096x4096x50 domain")
    ap.add_argument("--no-extras", action="store_true",
                    help="with c5: skip the 1024x1024x30 domain and its companions")
    ap.add_argument("--no-small", action="store_true", help="skip the launch-bound small case")
    ap.add_argument("--no-ensemble", action="store_true", help="skip the 48-domain ensemble")
    ap.add_argument("--no-std", action="store_true",
                    help="skip the standard scheme (RK3 + WRF limiter) measurement")
    ap.add_argument("--no-handoff", action="store_true",
                    help="skip the host transfer and snapshot measurement")
    ap.add_argument("--no-wind", action="store_true",
                    help="skip the wind-balance, dt and forcing kernels' timing")
    ap.add_argument("--nx", type=int, default=1024)
    ap.add_argument("--ny", type=int, default=1024)
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU; --gpus {args.gpus} is not supported "
              "(the library runs one domain or ensemble per GPU; the decomposition over "
              "several GPUs is designed but not implemented)", file=sys.stderr)
        return 2
    if args.workload == "c2":
        out = c2_line(args, cpu=not args.no_cpu)
    else:
        out = c5_line(args)
        if not args.no_extras:
            log("the 1024x1024x30, 10-species domain and its companions ...")
            c2 = c2_line(args, cpu=False)
            for k in ("metric", "unit", "n_gpus", "steps", "warmup", "higher_is_better",
                      "scaling", "vs_baseline", "data"):
                c2.pop(k, None)
            out["c2_1024x1024x30"] = c2
    print(json.dumps(out), flush=True)
    return 0


def c2_line(args, cpu: bool) -> dict:
    """The 1024x1024x30, 10-species domain at mpdata_order 3 + FCT in its
    variants (the best bit-exact one as the value), and its companions."""
    from hicar_amd import synthetic
    log("generating the 1024x1024x30, 10-species workload ...")
    case = synthetic.config2(nx=args.nx, ny=args.ny)
    d = case.domain
    S = len(d.species)
    cells = d.nx * d.ny * d.nz
    variants = {"plain": 0, "batched": 1, "batched_bf16": 1}
    todo = list(variants) if args.variant == "all" else [args.variant]
    results = {}
    for name in todo:
        log(f"variant {name}: {args.warmup} warmup + {args.steps} timed steps ...")
        if name == "batched_bf16":
            set_bf16(case)
        t, stats = measure(case, variants[name], args.steps, args.warmup)
        lc = stats.pop("_launch_config", None)
        results[name] = {"seconds": t, "value": cells * S * args.steps / t, "stats": stats,
                         "b_step": step_bytes(d), "launch_config": lc}
        log(f"  {name}: {results[name]['value'] / 1e9:.2f} G cell-species/s, "
            f"{1e3 * t / args.steps:.2f} ms/step")
    wind = None
    if args.variant == "all" and not args.no_wind:
        wind = measure_wind_steps(case)
        log("  wind steps: " + ", ".join(f"{k} {v['avg_ms']:.3f} ms ({v['achieved_GBps']:.0f} GB/s)"
                                         for k, v in wind.items()))
    # launch-bound small domain: eager vs graph replay
    small = {}
    if args.variant == "all" and not args.no_small:
        c1 = synthetic.config1()
        c1.options.adv_options.MPDATA_FCT = True
        n1 = c1.domain.nx * c1.domain.ny * c1.domain.nz * len(c1.domain.species)
        for g in (False, True):
            t, _ = measure(c1, 1, 100, 10, profile=False, graph=g)
            small["graph" if g else "eager"] = n1 * 100 / t
        log(f"  256x64x20 ridge, 1 species, batched: eager {small['eager'] / 1e9:.2f}, "
            f"graph {small['graph'] / 1e9:.2f} G cell-species/s")
    ensemble = None
    if args.variant == "all" and not args.no_ensemble:
        log("48-domain ensemble (6 species, order 2 + FCT): generating inputs ...")
        ensemble = measure_ensemble(args.steps, args.warmup)
        log(f"  ensemble of 48: eager {ensemble['eager']['value'] / 1e9:.2f}, graph "
            f"{ensemble['graph']['value'] / 1e9:.2f} G cell-species/s")
    handoff = None
    if args.variant == "all" and not args.no_handoff:
        handoff = measure_host_handoff(case, min(args.steps, 10), args.warmup)
        log(f"  host hand-off: species upload {handoff['upload_ms']:.1f} ms "
            f"({handoff['upload_GBps']:.1f} GB/s), download {handoff['download_ms']:.1f} ms "
            f"({handoff['download_GBps']:.1f} GB/s); step {handoff['step_ms']:.2f} ms, "
            f"{handoff['step_ms_while_snapshot_in_flight']:.2f} ms while a snapshot is copied "
            f"out ({handoff['snapshot_to_host_ms']:.0f} ms to the host arrays)")
    std = None
    if args.variant == "all" and not args.no_std:
        log("standard scheme (h5/v3, WRF limiter, RK3), same domain: generating inputs ...")
        std = measure_std(args.nx, args.ny, args.steps, args.warmup)
        log(f"  standard scheme: {std['value'] / 1e9:.2f} G cell-species/s, "
            f"{std['ms_per_step']:.2f} ms/step")
    exact_ok = [k for k in results if k in ("plain", "batched")]
    best = max(exact_ok or results, key=lambda k: results[k]["value"])
    r = results[best]
    stats = r["stats"]
    # compulsory bytes of one step (inputs read once, every species read and
    # written once at its storage width): 4*(5*N + 2*N_u + 2*N_v) + sum_s 2*b_s*N
    b_step = r["b_step"]
    per_unit = b_step / (cells * S)  # bytes per cell-species update
    dom_k = max(stats, key=lambda k: stats[k]["total_ms"])
    ks = stats[dom_k]
    avg_s = ks["total_ms"] / ks["launches"] / 1e3
    # cell-species one launch of the dominant kernel advances: all species for
    # the batched kernels and the Courant kernel, one species otherwise
    units = cells * (S if (best != "plain" or dom_k == "courant") else 1)
    achieved = per_unit * units / avg_s
    traffic = read_traffic(KERNEL_SYMBOL.get(dom_k, dom_k))
    roofline = {"bound": "hbm", "achieved": achieved / 1e9, "peak": HBM_PEAK / 1e9,
                "unit": "GB/s", "frac": achieved / HBM_PEAK, "traffic": traffic,
                "kernel": dom_k, "avg_launch_ms": avg_s * 1e3,
                "bytes_per_cell_species": per_unit, "cell_species_per_launch": units,
                "kernel_own_bytes_per_launch": ks["alg_bytes"] / ks["launches"]}
    # the kernel's other roof: VALU issue (instruction count per launch from
    # the committed SQ_INSTS_VALU profile, over the live launch duration)
    vi = read_valu(KERNEL_SYMBOL.get(dom_k, dom_k))
    if vi is not None and best != "plain":
        roofline["valu"] = {"wave_instr_per_launch": vi, "achieved": vi / avg_s / 1e9,
                            "peak": VALU_ISSUE_PEAK / 1e9, "unit": "G wave-instr/s",
                            "frac": vi / avg_s / VALU_ISSUE_PEAK}
    out = {
        "metric": "MPDATA cell-species updates/s & % HBM roofline, plain FP32 vs batched/mixed",
        "value": r["value"],
        "unit": "cell-species updates/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": 1e3 * r["seconds"] / args.steps,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "parity": "bit-identical to the FP32 oracle (plain and batched)",
        "data": "synthetic",
        "config": {"workload": f"single domain {d.nx}x{d.ny}x{d.nz}, {S} species, "
                               "mpdata_order 3 + FCT, advect_density, Courant 0.5",
                   "variants_run": todo,
                   "nx": d.nx, "ny": d.ny, "nz": d.nz, "species": S, "mpdata_order": 3,
                   "fct": True, "variant": best, "dt": case.dt},
        "roofline": roofline,
        "variants": {k: {"value": v["value"], "ms_per_step": 1e3 * v["seconds"] / args.steps,
                         "compulsory_hbm_fraction": v["b_step"] * args.steps / v["seconds"] / HBM_PEAK,
                         "launch_config": v["launch_config"] if variants[k] == 1 else None,
                         "kernels": {kk: {"avg_ms": s["total_ms"] / s["launches"],
                                          "launches": s["launches"],
                                          "achieved_GBps": s["alg_bytes"] / s["total_ms"] / 1e6}
                                     for kk, s in v["stats"].items()}}
                     for k, v in results.items()},
        "compulsory_hbm_fraction": b_step * args.steps / r["seconds"] / HBM_PEAK,
        "launch_bound_256x64x20": small,
        "ensemble_48": ensemble,
        "standard_scheme_rk3": std,
        "host_handoff": handoff,
        "wind_steps": wind,
    }
    if cpu:
        log("CPU baseline (oracle, one image per thread) ...")
        out["cpu_baseline"] = cpu_baseline(case)
    return out


if __name__ == "__main__":
    sys.exit(main())
