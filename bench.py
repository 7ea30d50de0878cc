"""Benchmark of the FDTD time step on one MI355X.

Workload: the large dielectric-sphere scene -- 512^3 cells + a 12-cell CPML
on all six faces (536^3 = 153,990,656 cells), sphere of radius 0.35 x edge
with eps_r drawn from U[2, 6] (seed 2024), Gaussian TFSF plane wave, 1 GHz
NF2FF box -- stepped in FP64 by the HIP engine.  A step is one full time
step (H pass + CPML, TFSF, E pass + CPML, TFSF, NF2FF accumulation) over the
whole grid; the metric is Yee cell-updates per second (cells x steps / s,
cells including the CPML, as the reference's benchmark counts them,
test/benchmark.cu:209-216).

The timed region is exactly --steps steps after --warmup untimed ones, with
fields, coefficients and tables already resident in HBM.  Per-kernel HIP
events recorded on the engine's stream inside that region give the average
duration of the dominant kernel, from which the roofline fraction is formed
with the algorithmic bytes of one launch.  The CPU baseline is the oracle
(a C restatement of the reference kernels, OpenMP over x) timed on a few
steps of the same scene on this host.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--precision fp64]
       python bench.py --workload batch   (64 uneven grids, FP32, batched kernels)
       python bench.py --workload precision --steps 4000   (FP64/FP32/BF16/BF16C far-field error)
       python bench.py --workload learned   (learned 2-cell layer: training, reflection, speed)
       python bench.py --workload nf2ff_td --n 256   (NF2FF time-domain accumulation cost)
       python bench.py --workload dispersive   (Drude + Lorentz sphere, FP64 vs FP32)
       python bench.py --workload cylinder2d   (2-D TMz PEC cylinder, FP64 vs FP32)
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

HBM_PEAK_GBPS = 8000.0  # MI355X HBM3E, published


def traffic_file(name: str, tuning: dict | None = None):
    """HBM bytes per launch from profiles/traffic_<name>.json (two rocprofv3
    counter runs, FETCH_SIZE and WRITE_SIZE, of the same workload), or None
    when there is no such file or it was taken at another tiling."""
    path = os.path.join(ROOT, "profiles", f"traffic_{name}.json")
    if not os.path.exists(path):
        return None
    with open(path) as f:
        rec = json.load(f)
    want = rec.get("tuning")
    if want and tuning is not None and any(tuning.get(k) != v for k, v in want.items()):
        return None
    return rec.get("hbm_bytes_per_launch")


def pml_bytes(sim, pass_name: str, cbytes: int) -> int:
    """Algorithmic CPML bytes of one pass: for every psi element updated,
    read psi, write psi, read c_psi (the four psi arrays of a face hold
    exactly the corrected ranges)."""
    import xfdtd_cuda_amd as xf
    names = ("ea_psi_hb", "eb_psi_ha") if pass_name == "e" else ("ha_psi_eb", "hb_psi_ea")
    total = 0
    for p in range(6):
        try:
            for n in names:
                total += sim.array(f"pml.{p}.{n}").size
        except xf.XFError:
            break
    return total * 3 * cbytes


def main(argv=None) -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--precision", default=None, choices=["fp64", "fp32", "bf16", "bf16c", "fp16"],
                    help="default: fp64 for the sphere, fp32 for the batch")
    ap.add_argument("--n", type=int, default=512, help="interior cells per edge")
    ap.add_argument("--pml", type=int, default=12)
    ap.add_argument("--cpu-steps", type=int, default=5,
                    help="FP64 steps of each all-core CPU window (three windows, median; plus "
                         "three one-step single-thread windows), native build of the oracle")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-stream", action="store_true")
    ap.add_argument("--calib", action="store_true",
                    help="also run the plain-load copy kernel (2 GiB) before the steps, so a "
                         "counter run holds both copy kernels for the FETCH_SIZE scale")
    ap.add_argument("--workload", default="sphere",
                    choices=["sphere", "batch", "precision", "learned", "nf2ff_td",
                             "dispersive", "cylinder2d", "scenes"],
                    help="sphere: one 512^3 + CPML grid (default); batch: 64 uneven grids; "
                         "precision: the sphere run to the end in fp64, fp32, bf16 with "
                         "far-field errors against fp64; learned: the learned 2-cell layer "
                         "trained on the GPU, its reflection and step time against CPMLs; "
                         "nf2ff_td: the sphere with and without NF2FF time-domain boxes; "
                         "scenes: every quoted scene on the GPU and the CPU oracle")
    ap.add_argument("--tile-y", type=int, default=0, help="rows per Yee tile (0: engine default)")
    ap.add_argument("--chunks", type=int, default=0, help="marches along x (0: engine default)")
    ap.add_argument("--no-nt", action="store_true",
                    help="plain loads/stores for the updated field (sphere workload)")
    ap.add_argument("--k32", action="store_true",
                    help="32-lane k-tiles with two j-rows per wave (sphere workload)")
    ap.add_argument("--pml-streams", action="store_true",
                    help="CPML-free and CPML tiles of a pass in two launches on two streams "
                         "(sphere workload)")
    ap.add_argument("--xcd", action="store_true",
                    help="XCD-aware block order: each XCD takes a contiguous eighth of the tiles "
                         "(sphere workload)")
    ap.add_argument("--pml-ztail", action="store_true",
                    help="z-face CPML corrections at the end of each Yee tile instead of a launch "
                         "of their own (sphere workload)")
    ap.add_argument("--tfsf-ztail", action="store_true",
                    help="with --pml-ztail: the TF/SF corrections of the z = const faces applied "
                         "by the Yee tiles too (sphere workload)")
    ap.add_argument("--pml-fused", action="store_true",
                    help="z-face CPML corrections inside the Yee kernels instead of a launch of "
                         "their own (sphere workload)")
    ap.add_argument("--graph", action="store_true",
                    help="replay each step as a hipGraph (batch, precision, learned, scenes, "
                         "dispersive, cylinder2d); eager launches measured faster on MI355X "
                         "in all cases tried but the 536^3 sphere in FP32")
    ap.add_argument("--coeff", default="table", choices=["table", "dense"],
                    help="sphere workload: per-cell coefficient ids into a table (the compact "
                         "layout, default) or the reference's 18 per-cell coefficient arrays "
                         "streamed by the kernels (XF_COEFF_DENSE)")
    ap.add_argument("--td-boxes", type=int, default=3, help="NF2FF-TD boxes of nf2ff_td")
    ap.add_argument("--count", type=int, default=64, help="grids of the batch workload")
    ap.add_argument("--batch-tuning", default=None,
                    help="batch workload: fixed tiling 'tile_y,planes,k32,xcd' instead of the "
                         "autotuner (for counter runs)")
    ap.add_argument("--batch-only", action="store_true",
                    help="batch workload: time only the batch in the chosen precision (no "
                         "sequential, FP64 or learned-layer runs; for counter runs)")
    ap.add_argument("--full-steps", type=int, default=2000,
                    help="batch workload: steps of the full runs whose far fields are compared "
                         "(FP32 batch and the learned-layer batch against the FP64 batch; 0 skips)")
    args = ap.parse_args(argv)

    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py: this engine runs on one GPU; runs over several GPUs are not "
              "implemented (only --gpus 1 is accepted)", file=sys.stderr)
        return 2
    if args.workload == "batch":
        return bench_batch(args)
    if args.workload == "precision":
        return bench_precision(args)
    if args.workload == "learned":
        return bench_learned(args)
    if args.workload == "nf2ff_td":
        return bench_nf2ff_td(args)
    if args.workload in ("dispersive", "cylinder2d"):
        return bench_fp32_vs_fp64(args)
    if args.workload == "scenes":
        return bench_scenes(args)
    args.precision = args.precision or "fp64"

    import xfdtd_cuda_amd as xf
    from xfdtd_cuda_amd import _native, scenes

    if xf.device_count() < 1:
        print("bench.py: no HIP device", file=sys.stderr)
        return 1

    K, W = args.steps, args.warmup
    total_steps = W + K + (0 if args.no_cpu else 3 * args.cpu_steps + 3) + 1
    t_setup = time.perf_counter()
    dense = args.coeff == "dense"
    sim = scenes.large_sphere(n=args.n, pml=args.pml, steps=total_steps,
                              layout="dense" if dense else "compact")
    (nx, ny, nz), dt, _ = sim.info()
    cells = nx * ny * nz
    t_up = time.perf_counter()
    build_s = t_up - t_setup
    eng = xf.Engine(sim, precision=args.precision, timing=False,
                    coeff="dense" if dense else "auto").upload()
    upload_s = time.perf_counter() - t_up
    if args.tile_y or args.chunks or args.pml_fused or args.k32 or args.no_nt or args.pml_streams or \
            args.pml_ztail or args.tfsf_ztail or args.xcd:
        eng.set_tiling(args.tile_y or 1, args.chunks, xcd_remap=args.xcd, nontemporal=not args.no_nt,
                       pml_split=not args.pml_fused, k32=args.k32, pml_streams=args.pml_streams,
                       pml_ztail=args.pml_ztail, tfsf_ztail=args.tfsf_ztail)
    setup_s = time.perf_counter() - t_setup
    print(f"# setup {setup_s:.1f} s, grid {nx}x{ny}x{nz}, {eng.describe()}", file=sys.stderr,
          flush=True)

    copy_gbps = None
    if not args.no_stream:
        # one 16-byte element per lane, non-temporal: the fastest copy shape
        # measured on MI355X (grid-stride copy loops reach ~4.8 TB/s only)
        copy_gbps = _native.stream_bench(2 << 30, 10, 0, 6)
        print(f"# stream copy {copy_gbps:.0f} GB/s", file=sys.stderr, flush=True)
        if args.calib:
            plain = _native.stream_bench(2 << 30, 10, 0, 5)
            print(f"# plain-load copy {plain:.0f} GB/s", file=sys.stderr, flush=True)

    eng.run(W)
    eng.set_timing(True)
    eng.reset_timing()
    t0 = time.perf_counter()
    eng.run(K)  # synchronous: returns after the last event of the region
    wall = time.perf_counter() - t0
    tm = eng.timing()
    eng.set_timing(False)

    ms_per_step = tm["run_ms"] / K
    value = cells * K / (tm["run_ms"] * 1e-3) / 1e9  # Gcells/s
    sbytes = {"fp64": 8, "fp32": 4, "bf16": 2, "bf16c": 3, "fp16": 2}[args.precision]
    cbytes = 8 if args.precision == "fp64" else 4
    id_bytes = 1  # compact layout: uint8 material index (<= 256 materials)
    # dense: the uint8 id (dispersive flag) plus 9 coefficients per cell and pass
    per_cell_pass = 9 * sbytes + id_bytes + (9 * cbytes if dense else 0)
    bytes_h = cells * per_cell_pass + pml_bytes(sim, "h", cbytes)
    bytes_e = cells * per_cell_pass + pml_bytes(sim, "e", cbytes)
    h_ms = tm["yee_h_ms"] / tm["yee_h_launches"]
    e_ms = tm["yee_e_ms"] / tm["yee_e_launches"]
    if e_ms >= h_ms:
        kernel, avg_ms, alg_bytes = "k_yee_e3", e_ms, bytes_e
    else:
        kernel, avg_ms, alg_bytes = "k_yee_h3", h_ms, bytes_h
    one_pass = " step3=1" in eng.describe()
    if one_pass:  # H and E in one launch, timed as the E pass: 12 values and one id a cell
        kernel, avg_ms = "k_step3", e_ms
        alg_bytes = cells * (12 * sbytes + id_bytes) + pml_bytes(sim, "h", cbytes) + pml_bytes(sim, "e", cbytes)
    elif "pml_split=1" in eng.describe():
        kernel += "+k_pml_z"  # the pass: Yee kernel, then its z-face CPML launch
    achieved = alg_bytes / (avg_ms * 1e-3) / 1e9
    traffic = None
    tfile = os.path.join(ROOT, "profiles", f"traffic_{kernel.replace('+', '_')}_{args.precision}_{nx}"
                                           f"{'_dense' if dense else ''}.json")
    if os.path.exists(tfile):
        with open(tfile) as f:
            traffic = json.load(f).get("hbm_bytes_per_launch")

    t_dn = time.perf_counter()
    eng.download()  # fields, psi and NF2FF currents back into the host arrays
    download_s = time.perf_counter() - t_dn
    cpu = None
    if not args.no_cpu:
        cpu = cpu_baseline(sim, cells, args.cpu_steps, f"{nx}x{ny}x{nz}")
    eng.close()

    out = {
        "metric": "Yee cell-updates/s (Gcells/s) & % HBM roofline",
        "value": round(value, 4),
        "unit": "Gcells/s",
        "n_gpus": 1,
        "steps": K,
        "warmup": W,
        "ms_per_step": round(ms_per_step, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": {"fp64": "f64", "fp32": "f32", "bf16": "bf16-storage/f32",
                  "bf16c": "bf16+int8-residual-storage/f32", "fp16": "fp16-storage/f32"}[args.precision],
        "data": "synthetic",
        "config": {"workload": f"dielectric sphere {nx - 2 * args.pml}^3 + {args.pml}-cell CPML "
                               f"({nx}x{ny}x{nz} cells), TFSF + NF2FF 1 GHz, {args.precision}",
                   "cells": cells,
                   "layout": ("dense (18 per-cell coefficient arrays, "
                              f"{9 * cbytes} B per cell and pass)") if dense
                   else "compact (uint8 material index)",
                   "wall_s": round(wall, 4),
                   "end_to_end_s": {"scene_build": round(build_s, 2), "upload": round(upload_s, 2),
                                    "steps_timed": round(wall, 3), "download": round(download_s, 2)}},
        "roofline": {"bound": "hbm", "kernel": kernel, "achieved": round(achieved, 1),
                     "peak": HBM_PEAK_GBPS, "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBPS, 4),
                     "traffic": traffic, "alg_bytes_per_launch": alg_bytes,
                     "avg_launch_ms": round(avg_ms, 4),
                     "h_ms": round(h_ms, 4), "e_ms": round(e_ms, 4),
                     "measured_copy_GBps": round(copy_gbps, 1) if copy_gbps else None},
        "cpu_baseline": cpu,
    }
    print(json.dumps(out), flush=True)
    return 0


def cpu_baseline(sim, cells: int, steps: int, shape: str) -> dict:
    """The oracle (a C restatement of the reference kernels) built on this
    host with -march=native (no FP contraction), timed on the same scene:
    three all-core windows of `steps` steps and three one-step single-thread
    windows, medians."""
    import os as _os
    import oracle
    nthr = len(_os.sched_getaffinity(0)) if hasattr(_os, "sched_getaffinity") else _os.cpu_count()
    nthr = max(1, min(nthr, int(_os.environ.get("OMP_NUM_THREADS", nthr))))
    all_s = oracle.time_steps(sim.scene_ptr(), steps, nthr, 3)
    one_s = oracle.time_steps(sim.scene_ptr(), 1, 1, 3)
    med_all, med_one = float(np.median(all_s)), float(np.median(one_s))
    model = ""
    try:
        with open("/proc/cpuinfo") as f:
            model = next((ln.split(":", 1)[1].strip() for ln in f if ln.startswith("model name")), "")
    except OSError:
        pass
    return {"value": round(cells * steps / med_all / 1e9, 4), "unit": "Gcells/s", "cores": nthr,
            "kind": "port",
            "sample": f"{steps} FP64 steps of the same {shape} scene per window, median of 3 "
                      f"windows ({', '.join(f'{t:.2f}' for t in all_s)} s), oracle/xf_oracle.c "
                      f"built -O3 -march=native -ffp-contract=off, {nthr} OpenMP threads",
            "single_thread": round(cells / med_one / 1e9, 4),
            "single_thread_sample": f"1 step per window, median of 3 ({', '.join(f'{t:.2f}' for t in one_s)} s)",
            "cpu_model": model}


def bench_batch(args) -> int:
    """64 sphere grids of uneven sizes (edges U[48, 160] + 8-cell CPML,
    radius U[0.2, 0.4] x edge, eps_r U[1.5, 8], seed 7) stepped together in
    one persistent launch per Yee pass (eager launches, or a hipGraph with
    --graph), tile shape from the autotuner.  Besides the batch rate the
    line carries the same grids run one after another through the
    single-grid engine, and the batch in FP64, for the speed-ups batching and
    FP32 give."""
    import xfdtd_cuda_amd as xf
    from xfdtd_cuda_amd import scenes

    prec = args.precision or "fp32"
    K, W, KT = args.steps, args.warmup, 5
    steps_needed = W + K + KT + 8
    t0 = time.perf_counter()
    sims = scenes.batch_spheres(count=args.count, steps=max(steps_needed, 2 * K + 8))
    cells = sum(int(np.prod(s.info()[0])) for s in sims)
    print(f"# batch set-up {time.perf_counter() - t0:.1f} s, {len(sims)} grids, {cells} cells",
          file=sys.stderr, flush=True)

    def timed_batch(precision):
        b = xf.Batch(sims, precision=precision, use_graph=args.graph).upload()
        if args.batch_tuning:
            ty, planes, k32, xcd = (int(v) for v in args.batch_tuning.split(","))
            b.set_tuning(tile_y=ty, planes=planes, k32=bool(k32), xcd_remap=bool(xcd))
            best = b.tuning()
        else:
            best = b.autotune(trial_steps=3)
        b.run(W)
        b.reset_timing()
        b.run(K)
        run_ms = b.timing()["run_ms"]
        b.set_timing(True)
        b.reset_timing()
        b.run(KT)
        tm = b.timing()
        desc = b.describe()
        b.close()
        return run_ms, tm, best, desc

    run_ms, tm, best, desc = timed_batch(prec)
    print(f"# batch {prec}: {run_ms / K:.3f} ms/step, {desc}", file=sys.stderr, flush=True)
    value = cells * K / (run_ms * 1e-3) / 1e9
    if args.batch_only:
        h_ms = tm["yee_h_ms"] / tm["yee_h_launches"]
        e_ms = tm["yee_e_ms"] / tm["yee_e_launches"]
        print(json.dumps({"metric": "Yee cell-updates/s (Gcells/s) & % HBM roofline",
                          "value": round(value, 4), "unit": "Gcells/s", "steps": K, "warmup": W,
                          "ms_per_step": round(run_ms / K, 4), "batch_only": True, "describe": desc,
                          "h_ms": round(h_ms, 4), "e_ms": round(e_ms, 4)}), flush=True)
        return 0

    # the same grids one after another through the single-grid engine
    seq_ms = 0.0
    for s in sims:
        e = xf.Engine(s, precision=prec, use_graph=args.graph).upload()
        e.run(2)
        e.run(K)
        seq_ms += e.timing()["run_ms"]
        e.close()
    seq_value = cells * K / (seq_ms * 1e-3) / 1e9
    print(f"# sequential {prec}: {seq_ms / K:.3f} ms/step", file=sys.stderr, flush=True)

    run64, _, best64, _ = timed_batch("fp64")
    value64 = cells * K / (run64 * 1e-3) / 1e9
    print(f"# batch fp64: {run64 / K:.3f} ms/step", file=sys.stderr, flush=True)

    # the same spheres bounded by the 2-cell learned layer instead of the
    # 8-cell CPML, weights trained here on 16-cell CPML point-source runs
    from xfdtd_cuda_amd import learned
    smp, kmur = learned.record_samples(n=32, seeds=(0, 1, 2, 3, 4, 5), steps=300, every=2)
    w16, _ = learned.train_selected(smp, kmur)
    sims_cpml = sims
    sims = scenes.batch_spheres(count=args.count, steps=max(steps_needed, 2 * K + 8), pml=2,
                                lb_weights=w16.view(np.float16))
    cells_lb = sum(int(np.prod(s.info()[0])) for s in sims)
    run_lb, _, best_lb, _ = timed_batch(prec)
    print(f"# batch {prec} learned 2-cell layer: {run_lb / K:.3f} ms/step", file=sys.stderr, flush=True)
    sims = sims_cpml

    sbytes = {"fp64": 8, "fp32": 4, "bf16": 2, "bf16c": 3, "fp16": 2}[prec]
    cbytes = 8 if prec == "fp64" else 4
    bytes_h = sum(int(np.prod(s.info()[0])) * (9 * sbytes + 1) + pml_bytes(s, "h", cbytes)
                  for s in sims)
    bytes_e = sum(int(np.prod(s.info()[0])) * (9 * sbytes + 1) + pml_bytes(s, "e", cbytes)
                  for s in sims)
    h_ms = tm["yee_h_ms"] / tm["yee_h_launches"]
    e_ms = tm["yee_e_ms"] / tm["yee_e_launches"]
    if e_ms >= h_ms:
        kernel, avg_ms, alg_bytes = "k_yee_e3_batch", e_ms, bytes_e
    else:
        kernel, avg_ms, alg_bytes = "k_yee_h3_batch", h_ms, bytes_h
    if " step3=1" in desc:  # H and E in one launch, timed as the E pass
        kernel, avg_ms = "k_step3", e_ms
        alg_bytes = sum(int(np.prod(s.info()[0])) * (12 * sbytes + 1) + pml_bytes(s, "h", cbytes) +
                        pml_bytes(s, "e", cbytes) for s in sims)
    achieved = alg_bytes / (avg_ms * 1e-3) / 1e9

    accuracy = batch_far_field(args, prec, w16) if args.full_steps > 0 else None

    cpu = None
    if not args.no_cpu:
        import oracle
        threads = oracle.threads()
        tc = time.perf_counter()
        for s in sims:
            oracle.run(s.scene_ptr(), 1)
        cpu_s = time.perf_counter() - tc
        cpu = {"value": cells / cpu_s / 1e9, "unit": "Gcells/s", "cores": threads, "kind": "port",
               "sample": f"1 FP64 step of each of the {len(sims)} grids ({cpu_s:.1f} s), "
                         f"oracle/xf_oracle.c with {threads} OpenMP threads"}

    out = {
        "metric": "Yee cell-updates/s (Gcells/s) & % HBM roofline",
        "value": round(value, 4), "unit": "Gcells/s", "n_gpus": 1, "steps": K, "warmup": W,
        "ms_per_step": round(run_ms / K, 4), "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None,
        "dtype": {"fp64": "f64", "fp32": "f32", "bf16": "bf16-storage/f32",
                  "bf16c": "bf16+int8-residual-storage/f32", "fp16": "fp16-storage/f32"}[prec],
        "data": "synthetic",
        "config": {"workload": f"batch of {len(sims)} sphere grids, edges U[48,160] + 8-cell CPML "
                               f"({cells} cells), TFSF + NF2FF, {prec}, one persistent launch "
                               "per pass, " + ("hipGraph step" if args.graph else "eager launches"),
                   "cells": cells, "tuning": best, "describe": desc,
                   "sequential_single_grid_gcells": round(seq_value, 4),
                   "batch_speedup_vs_sequential": round(value / seq_value, 3),
                   "fp64_batch_gcells": round(value64, 4),
                   "learned2_boundary": {
                       "ms_per_step": round(run_lb / K, 4), "cells": cells_lb,
                       "speedup_vs_cpml8_same_spheres": round(run_ms / run_lb, 3),
                       "tuning": best_lb},
                   "speedup_vs_fp64": round(value / value64, 3), "fp64_tuning": best64,
                   "far_field_accuracy": accuracy},
        "roofline": {"bound": "hbm", "kernel": kernel, "achieved": round(achieved, 1),
                     "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                     "frac": round(achieved / HBM_PEAK_GBPS, 4),
                     "traffic": (traffic_file(f"{kernel}_{prec}_64grids", best)
                                 if kernel == "k_yee_e3_batch" and len(sims) == 64 else None),
                     "alg_bytes_per_launch": alg_bytes, "avg_launch_ms": round(avg_ms, 4),
                     "h_ms": round(h_ms, 4), "e_ms": round(e_ms, 4)},
        "cpu_baseline": cpu,
    }
    print(json.dumps(out), flush=True)
    return 0


def bench_precision(args) -> int:
    """The 512^3 + 12-cell CPML sphere stepped --steps steps (4000 for the
    full study) in FP64, FP32, BF16-storage/FP32-compute, compensated BF16
    storage (bf16 + an 8-bit residual per value)/FP32-compute and
    FP16-storage/FP32-compute.  Each mode's
    bistatic RCS at 1 GHz on the xz and yz cuts (360 angles) is compared with
    the FP64 run's: relative L2 error over the cut and the largest dB
    difference.  NF2FF sums are FP64 in every mode."""
    import xfdtd_cuda_amd as xf
    from xfdtd_cuda_amd import scenes

    S = args.steps
    theta = np.linspace(-np.pi, np.pi, 360)
    res = {}
    for prec in ("fp64", "fp32", "bf16", "bf16c", "fp16"):
        t0 = time.perf_counter()
        sim = scenes.large_sphere(n=args.n, pml=args.pml, steps=S, layout="compact")
        (nx, ny, nz), _, _ = sim.info()
        eng = xf.Engine(sim, precision=prec, use_graph=args.graph).upload()
        eng.run(S)
        run_ms = eng.timing()["run_ms"]
        eng.download()
        eng.close()
        inc = sim.incident_spectrum(1e9)
        rcs = [sim.far_field(0, 0, theta, phi, inc)[2] for phi in (0.0, np.pi / 2)]
        cells = nx * ny * nz
        res[prec] = {"gcells": cells * S / (run_ms * 1e-3) / 1e9, "ms_per_step": run_ms / S,
                     "rcs": rcs}
        print(f"# {prec}: {run_ms / S:.3f} ms/step over {S} steps "
              f"({time.perf_counter() - t0:.0f} s with set-up)", file=sys.stderr, flush=True)
        del sim

    def err(a, b):
        rel = float(np.linalg.norm(a - b) / np.linalg.norm(b))
        db = float(np.max(np.abs(10 * np.log10(np.maximum(a, 1e-30))
                                 - 10 * np.log10(np.maximum(b, 1e-30)))))
        return rel, db

    modes = {}
    for prec in ("fp64", "fp32", "bf16", "bf16c", "fp16"):
        r = res[prec]
        e = [err(r["rcs"][c], res["fp64"]["rcs"][c]) for c in range(2)]
        modes[prec] = {"gcells": round(r["gcells"], 4), "ms_per_step": round(r["ms_per_step"], 4),
                       "speedup_vs_fp64": round(r["gcells"] / res["fp64"]["gcells"], 3),
                       "rcs_rel_l2_xz": e[0][0], "rcs_rel_l2_yz": e[1][0],
                       "rcs_max_db_diff": max(e[0][1], e[1][1])}
    cells = (args.n + 2 * args.pml) ** 3
    out = {
        "metric": "Yee cell-updates/s (Gcells/s) & % HBM roofline",
        "value": modes["fp32"]["gcells"], "unit": "Gcells/s", "n_gpus": 1, "steps": S,
        "warmup": 0, "ms_per_step": modes["fp32"]["ms_per_step"], "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": f"precision study: sphere {args.n}^3 + {args.pml}-cell CPML "
                               f"({cells} cells), {S} steps per mode, RCS at 1 GHz vs FP64",
                   "modes": modes},
        "roofline": None, "cpu_baseline": None,
    }
    print(json.dumps(out), flush=True)
    return 0


def _rcs_cut(sim, phi: float, n: int = 360) -> np.ndarray:
    """RCS over n angles of theta in the phi plane at 1 GHz (the box's
    first frequency), normalised by the incident spectrum."""
    angles = np.linspace(-np.pi, np.pi, n)
    inc = sim.incident_spectrum(1e9)
    return np.asarray(sim.far_field(0, 0, angles, phi, inc)[2])


def batch_far_field(args, prec: str, w16) -> dict:
    """The accuracy condition of the batch: every grid of the
    batch run to the end (`--full-steps`) in `prec` and in FP64 (bit-identical
    to the oracle), and the same spheres bounded by the learned 2-cell layer
    instead of the 8-cell CPML; RCS (xz and yz cuts at 1 GHz) relative L2
    error of each grid against its FP64 CPML run, max and mean over grids."""
    import xfdtd_cuda_amd as xf
    from xfdtd_cuda_amd import scenes

    steps = args.full_steps
    t0 = time.perf_counter()

    def run(sims, precision, label):
        b = xf.Batch(sims, precision=precision).upload()
        b.autotune(trial_steps=2)
        ms = 0.0
        for _ in range(steps // 250):  # in pieces, so the run reports progress
            b.run(250)
            ms += b.timing()["run_ms"]
            print(f"#   {label}: {ms / 1e3:.1f} s of steps", file=sys.stderr, flush=True)
        if steps % 250:
            b.run(steps % 250)
            ms += b.timing()["run_ms"]
        b.download()
        b.close()
        return ms / steps

    def cuts(sims, label):
        # 72 angles per cut (every 5 degrees): the host far-field sum is the
        # slow part of this check
        out = []
        for q, s in enumerate(sims):
            out.append((_rcs_cut(s, 0.0, 72), _rcs_cut(s, np.pi / 2, 72)))
            if q % 16 == 15:
                print(f"#   {label}: far fields of {q + 1} grids", file=sys.stderr, flush=True)
        return out

    ref = scenes.batch_spheres(count=args.count, steps=steps)
    ms64 = run(ref, "fp64", "fp64")
    r64 = cuts(ref, "fp64")
    del ref
    red = scenes.batch_spheres(count=args.count, steps=steps)
    msr = run(red, prec, prec)
    rr = cuts(red, prec)
    del red
    lb = scenes.batch_spheres(count=args.count, steps=steps, pml=2, lb_weights=w16.view(np.float16))
    msl = run(lb, prec, "learned2")
    rl = cuts(lb, "learned2")
    del lb

    def errs(test):
        e = [max(float(np.linalg.norm(a - b) / np.linalg.norm(b)) for a, b in zip(t, r))
             for t, r in zip(test, r64)]
        return {"max": max(e), "mean": float(np.mean(e)), "median": float(np.median(e))}

    out = {"steps": steps, "reference": "the same grids in FP64 with the 8-cell CPML (the batch's FP64 "
                                        "results equal the oracle's bit for bit)",
           f"{prec}_rcs_rel_l2": errs(rr), "learned2_rcs_rel_l2": errs(rl),
           "ms_per_step": {"fp64": round(ms64, 4), prec: round(msr, 4), "learned2": round(msl, 4)},
           "speedup_vs_fp64": {prec: round(ms64 / msr, 3), "learned2": round(ms64 / msl, 3)},
           "bar": 1e-3}
    print(f"# far fields after {steps} steps ({time.perf_counter() - t0:.0f} s): {out}", file=sys.stderr,
          flush=True)
    return out


def bench_learned(args) -> int:
    """The learned absorbing layer end to end on the GPU: training data from
    16-cell CPML point-source runs (seeds 0-5, 32^3 interior), training by
    the HIP trainer, reflection error against the 16-cell CPML averaged over
    four unseen seeds next to Mur and 2/4/8-cell CPMLs, and the step time of a 256^3
    interior bounded by the 2-cell layer against the same interior with an
    8-cell CPML (FP32 fields)."""
    import xfdtd_cuda_amd as xf
    from xfdtd_cuda_amd import learned, scenes

    t0 = time.perf_counter()
    smp, k = learned.record_samples(n=32, seeds=(0, 1, 2, 3, 4, 5), steps=300, every=2)
    t_rec = time.perf_counter() - t0
    t0 = time.perf_counter()
    # six inits at three input-noise levels, the layer chosen on validation
    # seeds 11-13 (neither trained on nor judged)
    w16, cand = learned.train_selected(smp, k, inits=range(6), noises=(0.005, 0.01, 0.02))
    chosen = min(cand, key=lambda r: r["val_mean"])
    loss1 = chosen["loss"]
    t_train = time.perf_counter() - t0
    # the judge: four unseen seeds (40^3 interior, 400 steps); one seed alone
    # varies too much from scene to scene to rank boundaries
    judge_seeds = (7, 8, 9, 10)
    per_seed = {s: learned.reflection_errors(w16, seed=s, variants=[("learned", 2), ("mur", 2), ("cpml", 2),
                                                                      ("cpml", 4), ("cpml", 8)])
                for s in judge_seeds}
    err = {k2: float(np.mean([per_seed[s][k2] for s in judge_seeds])) for k2 in per_seed[judge_seeds[0]]}
    print(f"# {smp.shape[0]} samples in {t_rec:.1f} s, {len(cand)} layers trained and validated in "
          f"{t_train:.1f} s, chosen noise {chosen['noise']} init {chosen['init']} (validation mean "
          f"{chosen['val_mean']:.4g}), mean reflection over seeds {judge_seeds}: "
          f"{ {k2: round(v, 6) for k2, v in err.items()} }", file=sys.stderr, flush=True)

    K, W, n = args.steps, args.warmup, 256
    rates = {}
    for kind, size in (("learned", 2), ("cpml", 8)):
        sim = scenes.point_source_box(n=n, boundary=kind, size=size, steps=W + K + 4, seed=7,
                                      weights=w16 if kind == "learned" else None)
        cells = int(np.prod(sim.info()[0]))
        e = xf.Engine(sim, precision="fp32", use_graph=args.graph).upload()
        e.run(W)
        e.reset_timing()
        e.run(K)
        ms = e.timing()["run_ms"] / K
        e.close()
        rates[kind] = (cells, ms)
        print(f"# {kind}{size}: {cells} cells, {ms:.3f} ms/step", file=sys.stderr, flush=True)
    cells_l, ms_l = rates["learned"]
    cells_c, ms_c = rates["cpml"]
    out = {
        "metric": "Yee cell-updates/s (Gcells/s) & % HBM roofline",
        "value": round(cells_l / (ms_l * 1e-3) / 1e9, 4), "unit": "Gcells/s", "n_gpus": 1,
        "steps": K, "warmup": W, "ms_per_step": round(ms_l, 4), "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f32 fields, fp16-weight/fp32 network",
        "data": "synthetic",
        "config": {"workload": f"{n}^3 vacuum interior with seeded point sources bounded by the "
                               "learned 2-cell layer (vs an 8-cell CPML)",
                   "cells_learned": cells_l, "cells_cpml8": cells_c,
                   "ms_per_step_cpml8": round(ms_c, 4),
                   "interior_speedup_vs_cpml8": round(ms_c / ms_l, 3),
                   "reflection_vs_cpml16_mean": err,
                   "reflection_vs_cpml16_per_seed": {str(sd): {k2: float(v) for k2, v in r.items()}
                                                     for sd, r in per_seed.items()},
                   "training": {"samples": int(smp.shape[0]), "record_s": round(t_rec, 2),
                                "train_and_select_s": round(t_train, 2), "loss_after": loss1,
                                "selection": "lowest mean closed-loop reflection on validation "
                                             "seeds 11-13 over the candidates",
                                "chosen": {"noise": chosen["noise"], "init": chosen["init"]},
                                "candidates": cand}},
        "roofline": None, "cpu_baseline": None,
    }
    print(json.dumps(out), flush=True)
    return 0


def bench_fp32_vs_fp64(args) -> int:
    """Two of the reference's scenes run to the end in FP64 and in FP32, with
    the FP32 far field (and probe series) compared to the FP64 run's.
      dispersive: Drude core + one-pole Lorentz shell, 256^3 + 10-cell CPML,
        6000 steps, RCS at 0.5 / 1 / 2 GHz on the xz and yz cuts; the pole
        recursions (J) and NF2FF sums stay FP64 in the FP32 mode.
      cylinder2d: 2-D TMz PEC cylinder, 1000^2 + 10-cell CPML, dl = 1 mm,
        4000 steps, far field at 1 GHz over 360 angles in the xy plane and
        Ez probe series at three points.
    --steps overrides the step count (the default 100 means the full run)."""
    import tempfile

    import xfdtd_cuda_amd as xf
    from xfdtd_cuda_amd import scenes

    two_d = args.workload == "cylinder2d"
    steps = (4000 if two_d else 6000) if args.steps == 100 else args.steps
    n = (1000 if two_d else 256) if args.n == 512 else args.n
    angles = np.linspace(-np.pi, np.pi, 360)
    res = {}
    for prec in ("fp64", "fp32"):
        t0 = time.perf_counter()
        if two_d:
            sim = scenes.cylinder_2d(n=n, pml=10, steps=steps, init=False)
            for q, (fx, fy) in enumerate(((0.3, 0.0), (-0.25, 0.2), (0.0, -0.4))):
                half = n * 1e-3 / 2
                sim.add_movie_monitor("ez", (fx * 2 * half, fy * 2 * half, -np.inf), (1e-3, 1e-3, np.inf), 1)
            sim.init(steps)
            freqs = [1e9]
        else:
            sim = scenes.dispersive_sphere(n=n, pml=10, steps=steps)
            freqs = [0.5e9, 1e9, 2e9]
        (nx, ny, nz), _, _ = sim.info()
        eng = xf.Engine(sim, precision=prec, use_graph=args.graph).upload()
        # all but the last 10 steps untimed per kernel, the last 10 with
        # per-pass HIP events (the roofline's average pass time)
        eng.run(steps - 10)
        run_ms = eng.timing()["run_ms"]
        eng.set_timing(True)
        eng.reset_timing()
        eng.run(10)
        tm = eng.timing()
        run_ms += tm["run_ms"]
        desc = eng.describe()
        eng.download()
        eng.close()
        out = {"gcells": nx * ny * nz * steps / (run_ms * 1e-3) / 1e9, "ms_per_step": run_ms / steps}
        sb = 8 if prec == "fp64" else 4
        cb = 8 if prec == "fp64" else 4
        ncell = nx * ny * nz
        # E pass: 3-D reads E3, H3 and writes E3 (9 values) + id; 2-D reads
        # Ez, Hx, Hy and writes Ez (4 values) + id; plus the CPML psi traffic
        e_bytes = ncell * ((4 if two_d else 9) * sb + 1) + pml_bytes(sim, "e", cb)
        e_ms = tm["yee_e_ms"] / tm["yee_e_launches"]
        kname = ("k_yee_e2" if two_d else
                 ("k_yee_e3+k_pml_z+k_ade_e3" if "pml_split=1" in desc else "k_yee_e3+k_ade_e3"))
        if " step3=1" in desc:  # H and E in one launch, timed (with the ADE kernel) as the E pass
            kname = "k_step3+k_ade_e3"
            e_bytes = ncell * (12 * sb + 1) + pml_bytes(sim, "h", cb) + pml_bytes(sim, "e", cb)
        out["roofline"] = {"bound": "hbm", "kernel": kname,
                           "achieved": round(e_bytes / (e_ms * 1e-3) / 1e9, 1), "peak": HBM_PEAK_GBPS,
                           "unit": "GB/s",
                           "frac": round(e_bytes / (e_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
                           "traffic": (None if two_d else
                                       traffic_file(f"{kname.replace('+', '_')}_{prec}_{nx}")),
                           "alg_bytes_per_launch": e_bytes,
                           "avg_launch_ms": round(e_ms, 5), "h_ms": round(tm["yee_h_ms"] / tm["yee_h_launches"], 5),
                           "post_h_ms": round(tm["tfsf_ms"] / 10, 5), "post_e_ms": round(tm["nf2ff_ms"] / 10, 5),
                           "note": ("E pass events (the Yee kernel with its CPML, plus the ADE kernel "
                                    "in 3-D, where one launch does H and E; on 2-D FP64/FP32 grids the TF/SF corrections run inside "
                                    "k_yee_h2/k_yee_e2); algorithmic bytes count the fields, ids and "
                                    "psi, not the ADE J arrays. post_h_ms / post_e_ms: what follows "
                                    "each pass (TF/SF launches where not fused, sources, NF2FF, movies)") }
        out["desc"] = desc
        with tempfile.TemporaryDirectory() as d:
            if two_d:
                sim.output_far_field(0, np.pi / 2, angles, "xy", d)
                cuts = ["xy"]
            else:
                sim.output_far_field(0, angles, 0.0, "xz", d)
                sim.output_far_field(0, angles, np.pi / 2, "yz", d)
                cuts = ["xz", "yz"]
            rcs = {}
            for c in cuts:
                et = np.load(os.path.join(d, c, "e_theta.npy"))
                ep = np.load(os.path.join(d, c, "e_phi.npy"))
                for fi, f in enumerate(freqs):
                    inc = sim.incident_spectrum(f)
                    rcs[(c, f)] = 4 * np.pi * (np.abs(et[fi] / inc) ** 2 + np.abs(ep[fi] / inc) ** 2)
        out["rcs"] = rcs
        if two_d:
            out["probes"] = [sim.movie(q).reshape(steps, -1)[:, 0].copy() for q in range(3)]
        res[prec] = out
        print(f"# {prec}: {run_ms / steps:.4f} ms/step over {steps} steps "
              f"({time.perf_counter() - t0:.0f} s with set-up)", file=sys.stderr, flush=True)
        del sim

    errs = {f"rcs_rel_l2_{c}_{f / 1e9:g}GHz": float(np.linalg.norm(res["fp32"]["rcs"][(c, f)] - r)
                                                   / np.linalg.norm(r))
            for (c, f), r in res["fp64"]["rcs"].items()}
    if two_d:
        for q in range(3):
            a, b = res["fp32"]["probes"][q], res["fp64"]["probes"][q]
            errs[f"probe{q}_rel_l2"] = float(np.linalg.norm(a - b) / np.linalg.norm(b))
    cells = (n + 20) ** (2 if two_d else 3)
    out = {
        "metric": "Yee cell-updates/s (Gcells/s) & % HBM roofline",
        "value": round(res["fp32"]["gcells"], 4), "unit": "Gcells/s", "n_gpus": 1, "steps": steps,
        "warmup": 0, "ms_per_step": round(res["fp32"]["ms_per_step"], 5), "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": ("2-D TMz PEC cylinder" if two_d else "Drude + Lorentz sphere") +
                               f" {n}^{2 if two_d else 3} + 10-cell CPML ({cells} cells), "
                               f"{steps} steps, FP32 against FP64",
                   "fp64_gcells": round(res["fp64"]["gcells"], 4),
                   "speedup_vs_fp64": round(res["fp32"]["gcells"] / res["fp64"]["gcells"], 3),
                   "errors_vs_fp64": errs,
                   "max_error": max(errs.values())},
        "roofline": res["fp32"]["roofline"], "roofline_fp64": res["fp64"]["roofline"],
        "cpu_baseline": None,
    }
    print(json.dumps(out), flush=True)
    return 0


def bench_scenes(args) -> int:
    """Every scene the engine is quoted on, each timed on the GPU in FP64 and
    in its reduced-precision modes, and on the CPU oracle with one thread and
    with all threads:
      sphere156: dielectric sphere 140^3 + 8-cell CPML, 2400 steps;
      cylinder2d: 2-D TMz PEC cylinder 1000^2 + 10-cell CPML, 4000 steps;
      sphere536: sphere 512^3 + 12-cell CPML (a 400-step window of 4000);
      dispersive: Drude + Lorentz sphere 256^3 + 10-cell CPML, 6000 steps;
      batch: 64 sphere grids, edges U[48, 160] + 8-cell CPML (a 400-step
        window of 2000, tile shape from the autotuner).
    The GPU runs whole step counts where the scene is small and windows where
    it is large; the CPU runs windows sized to a few seconds (stated per row),
    starting from the GPU's final FP64 state."""
    import oracle
    import xfdtd_cuda_amd as xf
    from xfdtd_cuda_amd import scenes

    nthr = oracle.threads()
    specs = [
        ("sphere156", "dielectric sphere 140^3 + 8-cell CPML",
         lambda st: scenes.dielectric_sphere(n=140, pml=8, steps=st), 2400, ("fp64", "fp32"), 10, 200),
        ("cylinder2d", "2-D TMz PEC cylinder 1000^2 + 10-cell CPML",
         lambda st: scenes.cylinder_2d(n=1000, pml=10, steps=st), 4000, ("fp64", "fp32"), 40, 800),
        ("sphere536", "dielectric sphere 512^3 + 12-cell CPML",
         lambda st: scenes.large_sphere(n=512, pml=12, steps=st, layout="compact"), 400,
         ("fp64", "fp32", "bf16", "bf16c", "fp16"), 1, 5),
        ("dispersive", "Drude + Lorentz sphere 256^3 + 10-cell CPML",
         lambda st: scenes.dispersive_sphere(n=256, pml=10, steps=st), 6000, ("fp64", "fp32"), 2, 20),
    ]
    rows = []

    def cpu_windows(ptr_list, cells, c1, cn):
        out = {}
        for thr, steps in ((1, c1), (nthr, cn)):
            oracle.set_threads(thr)
            t0 = time.perf_counter()
            for p in ptr_list:
                oracle.run(p, steps)
            dt_s = time.perf_counter() - t0
            out[f"cpu_{'1thr' if thr == 1 else 'all'}"] = {
                "gcells": round(cells * steps / dt_s / 1e9, 5), "steps": steps, "threads": thr,
                "seconds": round(dt_s, 2)}
        oracle.set_threads(nthr)
        return out

    W = 3
    for name, what, build, gsteps, modes, c1, cn in specs:
        row = {"scene": name, "what": what}
        for prec in modes:
            extra = c1 + cn if prec == "fp64" else 0
            sim = build(W + gsteps + extra + 2)
            (nx, ny, nz), _, _ = sim.info()
            cells = nx * ny * nz
            eng = xf.Engine(sim, precision=prec, use_graph=args.graph).upload()
            eng.run(W)
            eng.run(gsteps)
            run_ms = eng.timing()["run_ms"]
            row["cells"] = cells
            row[f"gpu_{prec}"] = {"gcells": round(cells * gsteps / (run_ms * 1e-3) / 1e9, 4),
                                  "ms_per_step": round(run_ms / gsteps, 5), "steps": gsteps}
            if prec == "fp64":
                eng.download()
                eng.close()
                row.update(cpu_windows([sim.scene_ptr()], cells, c1, cn))
            else:
                eng.close()
            del sim
        for prec in modes[1:]:
            row[f"speedup_{prec}_vs_fp64"] = round(row[f"gpu_{prec}"]["gcells"] / row["gpu_fp64"]["gcells"], 3)
        row["gpu_fp64_vs_cpu_all"] = round(row["gpu_fp64"]["gcells"] / row["cpu_all"]["gcells"], 1)
        print(f"# {name}: {json.dumps(row)}", file=sys.stderr, flush=True)
        rows.append(row)

    # the batch of uneven grids
    K = 400
    row = {"scene": "batch", "what": "64 sphere grids, edges U[48,160] + 8-cell CPML"}
    for prec in ("fp64", "fp32"):
        extra = 2 if prec == "fp64" else 0
        sims = scenes.batch_spheres(count=64, steps=W + K + extra + 20)
        cells = sum(int(np.prod(s.info()[0])) for s in sims)
        b = xf.Batch(sims, precision=prec, use_graph=args.graph).upload()
        b.autotune(trial_steps=3)
        b.run(W)
        b.run(K)
        run_ms = b.timing()["run_ms"]
        row["cells"] = cells
        row[f"gpu_{prec}"] = {"gcells": round(cells * K / (run_ms * 1e-3) / 1e9, 4),
                              "ms_per_step": round(run_ms / K, 5), "steps": K}
        if prec == "fp64":
            b.download()
            b.close()
            row.update(cpu_windows([s.scene_ptr() for s in sims], cells, 1, 1))
        else:
            b.close()
        del sims
    row["speedup_fp32_vs_fp64"] = round(row["gpu_fp32"]["gcells"] / row["gpu_fp64"]["gcells"], 3)
    row["gpu_fp64_vs_cpu_all"] = round(row["gpu_fp64"]["gcells"] / row["cpu_all"]["gcells"], 1)
    print(f"# batch: {json.dumps(row)}", file=sys.stderr, flush=True)
    rows.append(row)

    big = next(r for r in rows if r["scene"] == "sphere536")
    out = {
        "metric": "Yee cell-updates/s (Gcells/s) & % HBM roofline",
        "value": big["gpu_fp64"]["gcells"], "unit": "Gcells/s", "n_gpus": 1,
        "steps": big["gpu_fp64"]["steps"], "warmup": W,
        "ms_per_step": big["gpu_fp64"]["ms_per_step"], "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f64", "data": "synthetic",
        "config": {"workload": "every quoted scene on the GPU (FP64 and reduced precision, "
                               + ("hipGraph" if args.graph else "eager launches")
                               + ") and on the CPU oracle (1 and all threads); value = the 536^3 sphere in FP64",
                   "scenes": rows},
        "roofline": None,
        "cpu_baseline": {"value": big["cpu_all"]["gcells"], "unit": "Gcells/s", "cores": nthr,
                         "kind": "port",
                         "sample": f"{big['cpu_all']['steps']} FP64 steps of the 536^3 sphere, "
                                   f"oracle/xf_oracle.c with {nthr} OpenMP threads"},
    }
    print(json.dumps(out), flush=True)
    return 0


def bench_nf2ff_td(args) -> int:
    """Cost of the NF2FF time-domain accumulation: the sphere scene (default
    here 256^3 + CPML) stepped with and without --td-boxes time-domain boxes
    on the frequency-domain box's surface, observation directions spread
    over the sphere.  The reference accumulates each face on one GPU thread
    (nf2ff_time_domain_data.cu:213-223); here every surface cell is a thread.
    The line reports the extra time per step and box and the surface cells
    per second it corresponds to."""
    import xfdtd_cuda_amd as xf
    from xfdtd_cuda_amd import scenes

    if xf.device_count() < 1:
        print("bench.py: no HIP device", file=sys.stderr)
        return 1
    prec = args.precision or "fp64"
    n = args.n if args.n != 512 else 256
    K, W = args.steps, args.warmup
    nb = max(1, args.td_boxes)
    dirs = [(float(np.arccos(1 - 2 * (q + 0.5) / nb)), float(2.399963 * q)) for q in range(nb)]
    runs = {}
    surface = 0
    for label, td in (("without", []), ("with", dirs)):
        sim = scenes.large_sphere(n=n, pml=args.pml, steps=W + K + 1, layout="compact", init=False)
        for th, ph in td:
            sim.add_nf2ff_td((args.pml + 3,) * 3, th, ph)
        sim.init(W + K + 1)
        if td:
            surface = sum(sim.array(f"nf2ff_td.0.{f}.prev.ea").size for f in xf.FACES)
            bins = sim.array("nf2ff_td.0.XN.wa").size
        eng = xf.Engine(sim, precision=prec).upload()
        eng.run(W)
        eng.reset_timing()
        eng.run(K)
        runs[label] = eng.timing()["run_ms"] / K
        eng.close()
        print(f"# {label} NF2FF-TD: {runs[label]:.4f} ms/step", file=sys.stderr, flush=True)
    (nx, ny, nz) = (n + 2 * args.pml,) * 3
    extra = (runs["with"] - runs["without"]) / nb
    out = {
        "metric": "NF2FF time-domain accumulation: extra ms per step and box",
        "value": round(extra, 5),
        "unit": "ms",
        "n_gpus": 1,
        "steps": K,
        "warmup": W,
        "ms_per_step": round(runs["with"], 4),
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": {"fp64": "f64", "fp32": "f32", "bf16": "bf16-storage/f32",
                  "bf16c": "bf16+int8-residual-storage/f32", "fp16": "fp16-storage/f32"}[prec],
        "data": "synthetic",
        "config": {"workload": f"dielectric sphere {n}^3 + {args.pml}-cell CPML ({nx}^3 cells), "
                               f"{nb} NF2FF-TD boxes of {surface} surface cells and {bins} bins",
                   "ms_per_step_without": round(runs["without"], 4),
                   "surface_cells_per_s": round(surface / (extra * 1e-3), 1) if extra > 0 else None},
    }
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
