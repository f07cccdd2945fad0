#!/usr/bin/env python3
"""Throughput of the central-slice hot path on one MI355X: 256^3 extraction + insertion, in slices/s.

One step = extract 4096 slices (256x129 complex64, "hc") from a 256^3 volume, then insert 10,000 CTF-weighted
slices (with CTF^2 weights) into a 256^3 volume + weights (FP32, LINEAR, windowed sinc of 1 voxel). Inputs
are synthetic (seeded) and already resident in HBM when the timed region starts.

Prints ONE JSON line (stdout): the metric, per-kernel achieved bandwidth against the MI355X HBM peak, and the
CPU baseline (the restated noa CPU path, timed on a bounded sample on this host).
"""
from __future__ import annotations

import argparse
import json
import os
import statistics
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

HBM_PEAK_GBS = 8000.0

PROFILES = ROOT / "profiles"


KERNELS = {
    "insert": {"one-wave": "insert_wave_kernel (+ insert_reduce_kernel)",
               "slab": "insert_slab_kernel (+ insert_reduce_kernel)"},
    "extract": {"block-copy gather": "extract_c32_kernel (+ brick_volume_kernel)",
                "row-major gather": "extract_c32_kernel",
                "LDS tiles": "extract_tile_kernel (+ extract_outside_kernel)"},
}


def measured_traffic(op: str, slices: int, variant: str):
    """HBM-side bytes per launch of an operator at the default workload, from the counter summary committed under
    profiles/ (a `traffic:` JSON line written with the FETCH_SIZE / WRITE_SIZE passes, scaled by the same counters on
    a 1 GiB device copy). The line records a hash of each kernel source it was measured with: when a source has
    changed since, the figure is stale and None is returned with the reason."""
    import hashlib
    for md in sorted(PROFILES.glob("*.md")):
        for line in md.read_text().splitlines():
            if not line.startswith("traffic: "):
                continue
            rec = json.loads(line[len("traffic: "):])
            if rec.get("op") != op or rec.get("slices") != slices or rec.get("variant") != variant:
                continue
            for src, digest in rec["sources"].items():
                now = hashlib.sha256((ROOT / src).read_bytes()).hexdigest()[:16]
                if now != digest:
                    return None, f"{md.name}: measured on another revision of {src}"
            nbytes = (rec["fetch_kib"] * rec["fetch_scale"] + rec["write_kib"] * rec["write_scale"]) * 1024
            return nbytes, md.name
    return None, "no counter summary for this operator and size"


METRIC = "slices/s and % HBM peak, 256\u00b3 insert+extract; p50/p99 request latency"


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def algorithmic_bytes_extract(b, n):
    """Output slices + volume + one Mat33 payload and one (y, x) f32 shift per slice (each read or written once);
    the phase shift is fused, so the slices are written once."""
    return b * n * (n // 2 + 1) * 8 + n * n * (n // 2 + 1) * 8 + b * 36 + b * 8


def algorithmic_bytes_insert(b, n):
    """c32 slices + f32 weights read once, c32 volume and f32 weights read and written once, Mat33 per slice."""
    px = n * (n // 2 + 1)
    vox = n * n * (n // 2 + 1)
    return b * px * (8 + 4) + 2 * vox * 8 + 2 * vox * 4 + b * 36


def cpu_cores() -> int:
    try:
        n = len(os.sched_getaffinity(0))
    except AttributeError:
        n = os.cpu_count() or 1
    return max(1, min(n, 16))   # at most 16 threads: the host cores that serve one GPU


def cpu_model() -> str:
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(ext, ins, n_ext_sample=64, n_ins_sample=48, full_insert=True, reps=5):
    """The oracle (noa's CPU algorithm restated, OpenMP) on the same inputs, under two thread settings:
    noa's heuristic, threads = min(cores, elements / 2^20) for the FULL workload (cpu/Iwise.hpp:104-116: all cores
    for the 4096-slice extraction, 8 for the 256^3 insertion), and all cores forced. Each leg: 1 warm-up run, then
    the median of `reps`. Extraction (+ phase shift) on the first `n_ext_sample` poses and insertion on the first
    `n_ins_sample` slices, extrapolated linearly (both costs are linear in the slice count); with `full_insert`, the
    whole 10,000-slice insertion is also run once under noa's heuristic, and the step uses that measurement."""
    sys.path.insert(0, str(ROOT / "oracle"))
    import numpy as np
    import oracle as O

    cores = cpu_cores()
    n = ext.volume.shape[1]
    vol = ext.volume.cpu().numpy()
    rot = ext.poses[:n_ext_sample]
    out = np.zeros((n_ext_sample, 1, n, n // 2 + 1), np.complex64)
    s = ins.slices[:n_ins_sample].cpu().numpy()
    w = ins.weights[:n_ins_sample].cpu().numpy()
    inv = np.ascontiguousarray(np.transpose(ins.poses[:n_ins_sample], (0, 2, 1)))

    def median_time(fn):
        fn()
        times = []
        for _ in range(reps):
            t0 = time.perf_counter()
            fn()
            times.append(time.perf_counter() - t0)
        return statistics.median(times)

    def extract(threads):
        O.extract_central_slices_3d("hc2hc", vol, None, (1, n, n, n), out, None, (n_ext_sample, 1, n, n), None, rot,
                                    n_threads=threads, force_threads=True)
        O.phase_shift_2d("hc2hc", out, out, (n_ext_sample, 1, n, n), ext.shifts[:n_ext_sample])

    def insert(threads):
        v = np.zeros((1, n, n, n // 2 + 1), np.complex64)
        wv = np.zeros((1, n, n, n // 2 + 1), np.float32)
        O.insert_central_slices_3d("h2h", s, w, (n_ins_sample, 1, n, n), v, wv, (1, n, n, n), None, inv,
                                   n_threads=threads, force_threads=True)

    n_e, n_i = ext.slice_shape[0], ins.slice_shape[0]
    settings = {
        "noa_heuristic": (min(cores, max(1, (n_e * n * (n // 2 + 1)) >> 20)), min(cores, max(1, (n * n * (n // 2 + 1)) >> 20))),
        "all_cores": (cores, cores),
    }
    legs = {}
    for name, (t_ext, t_ins) in settings.items():
        e = median_time(lambda: extract(t_ext)) / n_ext_sample
        i = median_time(lambda: insert(t_ins)) / n_ins_sample
        legs[name] = {"extract_threads": t_ext, "insert_threads": t_ins, "extract_ms_per_slice": e * 1e3,
                      "insert_ms_per_slice": i * 1e3, "slices_per_s": (n_e + n_i) / (e * n_e + i * n_i)}
        log(f"cpu {name}: extraction {e * 1e3:.3f} ms/slice ({t_ext} threads), insertion {i * 1e3:.2f} ms/slice "
            f"({t_ins} threads)")
    full = None
    if full_insert:
        t_ins = settings["noa_heuristic"][1]
        sl_all = ins.slices.cpu().numpy()
        w_all = ins.weights.cpu().numpy()
        inv_all = np.ascontiguousarray(np.transpose(ins.poses, (0, 2, 1)))
        v = np.zeros((1, n, n, n // 2 + 1), np.complex64)
        wv = np.zeros((1, n, n, n // 2 + 1), np.float32)
        t0 = time.perf_counter()
        O.insert_central_slices_3d("h2h", sl_all, w_all, (n_i, 1, n, n), v, wv, (1, n, n, n), None, inv_all,
                                   n_threads=t_ins, force_threads=True)
        full = time.perf_counter() - t0
        del sl_all, w_all, v, wv
        log(f"cpu full insertion of {n_i} slices: {full:.1f} s ({t_ins} threads)")
    h = legs["noa_heuristic"]
    ins_s = full if full is not None else h["insert_ms_per_slice"] * 1e-3 * n_i
    step_s = h["extract_ms_per_slice"] * 1e-3 * n_e + ins_s
    return {
        "value": (n_e + n_i) / step_s,
        "unit": "slices/s",
        "cores": max(settings["noa_heuristic"]),
        "kind": "port",
        "sample": (f"oracle (noa's CPU algorithm restated, OpenMP) with noa's thread heuristic: extraction + phase shift "
                   f"of {n_ext_sample} of the {n_e} poses extrapolated ({h['extract_threads']} threads), insertion of all "
                   f"{n_i} slices into 256^3 run once" if full is not None else
                   f"oracle with noa's thread heuristic: extraction of {n_ext_sample} poses and insertion of "
                   f"{n_ins_sample} slices, extrapolated") + f"; CPU: {cpu_model()}",
        "full_insert_s": full,
        "settings": legs,
    }


def _serving_calls(server, reqs):
    """Extraction and insertion calls of `reqs` with outputs carved from the server's pool (for tuning)."""
    from noa_amd import batch as nb
    ext, ins, off = [], [], 0
    for r in reqs:
        box, wr = r.box, r.box // 2 + 1
        if r.kind == "extract":
            out = server.pool.view(off, (r.count, 1, box, wr), torch_mod().complex64)
            off += r.output_bytes()
            ext.append(nb.extract_call("hc2hc", server.sources[box][r.volume], (1, box, box, box), out,
                                       (r.count, 1, box, box), r.rotations))
        else:
            v = server.pool.view(off, (1, box, box, wr), torch_mod().complex64)
            w = server.pool.view(off + (box * box * wr * 8 + 255) // 256 * 256, (1, box, box, wr), torch_mod().float32)
            off += r.output_bytes()
            ins.append(nb.insert_call("h2h", r.slices, r.weights, (r.count, 1, box, box), v, w, (1, box, box, box),
                                      r.rotations))
    return ext, ins


def torch_mod():
    import torch
    return torch


def serving_report(torch, dev, n_requests, qps_list, budget_gb=16.0, tune=True):
    """The mixed-box request stream through the continuous-batching server (noa_amd.serve: HBM-budgeted output
    pool, batches of extraction and insertion calls as persistent launches replayed from HIP graphs): p50/p99
    latency and served slices/s at each offered load of `qps_list` ("max": every request arrives at once, the
    device's capacity). Request inputs are on the device before each run; latency is completion (event passed)
    minus arrival. The batched kernels' grids and pixels per lane are autotuned first on a batch of the mix."""
    from noa_amd import autotune, serve, workloads
    from noa_amd import batch as nb
    import copy

    vols = workloads.serving_volumes(dev)
    base = workloads.serving_requests(dev, n_requests=n_requests, qps=1.0)
    server = serve.Server(vols, budget_bytes=int(budget_gb * (1 << 30)), n_streams=3, keep_results=False)
    for r in base:
        r.rotations = nb.nx.Mat33Array(r.rotations, device=dev)
    report = {"mix": "box {64,128,192,256,384} p {.3,.3,.2,.15,.05}; extract K~U{1..512} from 4 resident volumes "
                     "per box or insert K CTF-weighted slices into a per-request accumulator; Poisson arrivals",
              "requests": len(base), "extract_requests": sum(r.kind == "extract" for r in base),
              "insert_requests": sum(r.kind == "insert" for r in base), "budget_bytes": server.budget,
              "slots": len(server.slots), "path": "batched persistent launches (noa_hip_*_batch_*) replayed from HIP "
              "graphs, one batch per step"}
    if tune:
        sample = base[:32]
        ext, ins = _serving_calls(server, sample)
        slot = nb.BatchSlot(dev, graph=False)

        def run_ext():
            slot.prepare(ext, [])
            slot.upload()
            slot._launch()

        def run_ins():
            slot.prepare([], ins)
            slot.upload()
            slot._launch()
        best_e = autotune.tune("extract_batch", run_ext, reps=5, log=log)
        best_i = autotune.tune("insert_batch", run_ins, reps=5, log=log)
        report["tuning"] = {"extract_batch": {"pixels_per_lane": best_e.values[0], "workgroups": best_e.values[1],
                                              "ms": best_e.ms},
                            "insert_batch": {"workgroups": best_i.values[0], "ms": best_i.ms},
                            "sample": f"{len(ext)} extraction and {len(ins)} insertion calls of the mix in one batch"}
        del slot
    # Warm-up: the whole stream once at full load (insertion plans of every box and slice-count bucket).
    serve.run_open_loop(server, [_retimed(copy, r, 0.0) for r in base], timeout_s=300)
    torch.cuda.synchronize()
    sweep = []
    for qps in qps_list:
        reqs = [_retimed(copy, r, 0.0 if qps == "max" else r.arrival / float(qps)) for r in base]
        server.stats = serve.ServeStats()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        stats = serve.run_open_loop(server, reqs, timeout_s=300)
        torch.cuda.synchronize()
        wall = time.perf_counter() - t0
        row = {"qps": qps, "p50_ms": stats.percentile(50), "p99_ms": stats.percentile(99),
               "slices_per_s": stats.slices / wall, "wall_s": wall, "batches": stats.launches,
               "merged_requests": stats.merged, "mean_batch": len(reqs) / max(1, stats.launches)}
        sweep.append(row)
        log(f"serving qps={qps}: p50 {row['p50_ms']:.2f} ms, p99 {row['p99_ms']:.2f} ms, "
            f"{row['slices_per_s']:.0f} slices/s, {row['batches']} batches (mean {row['mean_batch']:.1f} requests)")
    report["sweep"] = sweep
    light = sweep[0]
    report.update({"p50_ms": light["p50_ms"], "p99_ms": light["p99_ms"], "qps": light["qps"],
                   "slices_per_s": light["slices_per_s"], "launches": light["batches"],
                   "merged_requests": light["merged_requests"]})
    return report


def _retimed(copy, r, arrival):
    c = copy.copy(r)
    c.arrival = arrival
    c.result = c.result_weight = None
    c.admitted = c.done = c.ready = c.offset = None
    return c


def precision_report(ext, nx, torch, n_ref=128):
    """Extraction from the 256^3 volume stored as FP32, FP16 pairs and BF16 pairs (FP32 math): rel-L2 and max error
    of each against the FP64 oracle (double volume and rotations) on the first n_ref poses, and the time of each for
    all poses."""
    sys.path.insert(0, str(ROOT / "oracle"))
    import numpy as np
    import oracle as O

    n = ext.volume.shape[1]
    b = ext.slice_shape[0]
    vol64 = ext.volume.cpu().numpy().astype(np.complex128)
    rot64 = ext.poses[:n_ref].astype(np.float64)
    ref = np.zeros((n_ref, 1, n, n // 2 + 1), np.complex128)
    O.extract_central_slices_3d("hc2hc", vol64, None, (1, n, n, n), ref, None, (n_ref, 1, n, n), None, rot64,
                                n_threads=cpu_cores(), force_threads=True)
    storages = {
        "fp32": ext.volume,
        "fp16": ext.volume.to(torch.complex32),
        "bf16": nx.ComplexBF16.from_complex(ext.volume),
    }
    out = torch.empty((b, 1, n, n // 2 + 1), dtype=torch.complex64, device=ext.volume.device)
    report = {"report": "extraction volume-storage precision", "config": "256^3 hc volume CN(0,1)*exp(-20|f|^2), "
              f"{b} uniform poses (error on the first {n_ref}), LINEAR, cutoff 0.5, FP32 math",
              "oracle": "FP64 restatement of noa's CPU extraction (double volume and rotations)"}
    for name, v in storages.items():
        def run():
            nx.extract_central_slices_3d("hc2hc", v, None, ext.volume_shape, out, None, ext.slice_shape, None,
                                         ext.rotations)
        run()
        torch.cuda.synchronize()
        got = out[:n_ref].cpu().numpy().astype(np.complex128)
        err = got - ref
        # Pixels on the cutoff circle (within 1e-3) can fall on either side in FP32 vs FP64 coordinates.
        fy = (np.arange(n) - n // 2)[:, None] / n
        fx = np.arange(n // 2 + 1)[None, :] / n
        inner = np.broadcast_to(np.abs(np.sqrt(fy ** 2 + fx ** 2) - 0.5) > 1e-3, err.shape)
        for _ in range(3):   # warm: the first calls of a storage also ramp the clocks and grow the memory pool
            run()
        t0 = torch.cuda.Event(enable_timing=True)
        t1 = torch.cuda.Event(enable_timing=True)
        t0.record()
        for _ in range(20):
            run()
        t1.record()
        torch.cuda.synchronize()
        report[name] = {
            "rel_l2": float(np.linalg.norm(err) / np.linalg.norm(ref)),
            "rel_l2_off_cutoff_circle": float(np.linalg.norm(err[inner]) / np.linalg.norm(ref[inner])),
            "max_abs": float(np.abs(err).max()),
            "max_abs_over_max_ref": float(np.abs(err).max() / np.abs(ref).max()),
            "volume_bytes": int(v.pairs.numel() * 2 if name == "bf16" else v.numel() * v.element_size()),
            "ms": t0.elapsed_time(t1) / 20,
        }
        log(f"{name}: rel-L2 {report[name]['rel_l2']:.3g}, max abs {report[name]['max_abs']:.3g}, "
            f"{report[name]['ms']:.3f} ms")
    return report


def neighbours_report(torch, dev, nx, ins, n, reps=5):
    """The steps on either side of the hot path, timed alone (not part of the step): the CTF prologue of the
    insertion (slice * CTF and CTF^2 in one pass over the insertion workload's raw spectra), an extraction from a
    virtual volume (a 61-view +-60 degree tilt series of 256^2 slices reprojected at 61 tilts offset by 1 degree),
    the rasterisation of 4096 slices and the isotropic CTF of a volume."""
    import numpy as np
    import noa_amd.signal as ns
    rep = {}
    b = ins.raw.shape[0]
    vals = torch.empty_like(ins.raw)
    wts = torch.empty((b, 1, n, n // 2 + 1), dtype=torch.float32, device=dev)

    def timed(fn, reps=reps):
        for _ in range(3):      # warm-up: plans, caches and the clocks reach their steady state
            fn()
        torch.cuda.synchronize()
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        ev[0].record()
        for _ in range(reps):
            fn()
        ev[1].record()
        torch.cuda.synchronize()
        return ev[0].elapsed_time(ev[1]) * 1e-3 / reps

    t = timed(lambda: ns.ctf_anisotropic_weighted("h2h", ins.raw, vals, wts, ins.slice_shape, ins.ctfs))
    nbytes = b * n * (n // 2 + 1) * (8 + 8 + 4) + b * 56
    dv = (vals - ins.slices).abs().max().item() / ins.slices.abs().max().item()
    rep["ctf_prologue"] = {
        "workload": f"{b} slices 256^2 (h2h): value * CTF and CTF^2, CTFAnisotropic<f32> per slice",
        "avg_ms": t * 1e3, "algorithmic_bytes": nbytes, "achieved_GBs": nbytes / t / 1e9,
        "frac_hbm_peak": nbytes / t / 1e9 / HBM_PEAK_GBS, "slices_per_s": b / t,
        "max_rel_diff_vs_workload_inputs": dv}
    log(f"ctf prologue: {t * 1e3:.3f} ms, {nbytes / t / 1e9:.0f} GB/s")
    del vals, wts

    tilts_in = np.deg2rad(np.arange(-60, 61, 2, dtype=np.float64))
    tilts_out = tilts_in + np.deg2rad(1.0)
    rin = np.stack([nx.euler2matrix([0.0, -a, 0.0], axes="zyx", dtype=np.float32) for a in tilts_in])
    rout = np.stack([nx.euler2matrix([0.0, a, 0.0], axes="zyx", dtype=np.float32) for a in tilts_out])
    b_in, b_out = len(tilts_in), len(tilts_out)
    src = ins.raw[:b_in]
    out = torch.empty((b_out, 1, n, n // 2 + 1), dtype=torch.complex64, device=dev)
    wout = torch.empty((b_out, 1, n, n // 2 + 1), dtype=torch.float32, device=dev)
    rin_d, rout_d = torch.from_numpy(rin).to(dev), torch.from_numpy(rout).to(dev)
    t = timed(lambda: nx.insert_and_extract_central_slices_3d(
        "h2h", src, None, (b_in, 1, n, n), out, wout, (b_out, 1, n, n), None, rin_d, None, rout_d))
    pairs = b_out * n * (n // 2 + 1) * b_in
    rep["virtual_volume"] = {
        "workload": f"insert_and_extract_central_slices_3d: {b_in} tilts (+-60, 2 deg) of 256^2 -> {b_out} tilts "
                    "offset by 1 deg, h2h, LINEAR, default windows",
        "avg_ms": t * 1e3, "output_slices_per_s": b_out / t, "pixel_slice_pairs_per_s": pairs / t,
        "nonzero_weight_fraction": (wout != 0).float().mean().item()}
    log(f"virtual volume: {t * 1e3:.3f} ms, {pairs / t / 1e9:.1f} G pixel-slice pairs/s")
    del out, wout

    # Rasterisation (trilinear scatter) of 4096 of the insertion workload's slices into a 256^3 volume + weights,
    # forward rotations (h2h, cutoff 0.5): the boxed kernel (sums of a box in LDS, one device-atomic flush per work
    # item), and once the one-lane-per-pixel kernel with device-wide float atomics for comparison.
    b_r = min(4096, b)
    rvol = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.complex64, device=dev)
    rw = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.float32, device=dev)
    fwd = torch.from_numpy(np.ascontiguousarray(ins.poses[:b_r])).to(dev)
    t = timed(lambda: nx.rasterize_central_slices_3d("h2h", ins.slices[:b_r], None, (b_r, 1, n, n), rvol, rw,
                                                     ins.volume_shape, None, fwd))
    prev = os.environ.get("NOA_HIP_RASTERIZE_LAYOUT")
    os.environ["NOA_HIP_RASTERIZE_LAYOUT"] = "direct"
    try:
        t_direct = timed(lambda: nx.rasterize_central_slices_3d("h2h", ins.slices[:b_r], None, (b_r, 1, n, n), rvol,
                                                                rw, ins.volume_shape, None, fwd), reps=1)
    finally:
        if prev is None:
            os.environ.pop("NOA_HIP_RASTERIZE_LAYOUT")
        else:
            os.environ["NOA_HIP_RASTERIZE_LAYOUT"] = prev
    px = b_r * n * (n // 2 + 1)
    rep["rasterize"] = {
        "workload": f"rasterize_central_slices_3d of {b_r} slices 256^2 into a 256^3 c32 volume + f32 weights (h2h, "
                    "cutoff 0.5)", "avg_ms": t * 1e3, "slices_per_s": b_r / t, "pixels_per_s": px / t,
        "kernel": "boxed (LDS sums per wave)", "direct_kernel_ms": t_direct * 1e3}
    log(f"rasterize {b_r} slices: {t * 1e3:.3f} ms (direct kernel {t_direct * 1e3:.1f} ms)")
    del rvol, rw, fwd

    # Insertion of a +-60 degree single-axis tilt series (10,000 slices, random in-plane angles; the same slices and
    # weights as the step): with the work plan of the uniform-orientation model, and with the pose-adaptive plan
    # (item order 3: passing slices counted on the device first).
    rng = np.random.default_rng(11)
    ang = np.stack([np.zeros(b), np.deg2rad(rng.uniform(-60, 60, b)), rng.uniform(0, 2 * np.pi, b)], -1)
    tilt = nx.euler2matrix(ang, axes="zyz", dtype=np.float32)
    tinv = torch.from_numpy(np.ascontiguousarray(np.transpose(tilt, (0, 2, 1)))).to(dev)
    tv = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.complex64, device=dev)
    tw = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.float32, device=dev)
    tilt_ms = {}
    prev = os.environ.get("NOA_HIP_INSERT_ORDER")
    try:
        for name, order in (("model_plan", "0"), ("pose_adaptive_plan", "3")):
            os.environ["NOA_HIP_INSERT_ORDER"] = order
            tilt_ms[name] = timed(lambda: nx.insert_central_slices_3d("h2h", ins.slices, ins.weights, ins.slice_shape,
                                                                      tv, tw, ins.volume_shape, None, tinv)) * 1e3
    finally:
        if prev is None:
            os.environ.pop("NOA_HIP_INSERT_ORDER")
        else:
            os.environ["NOA_HIP_INSERT_ORDER"] = prev
    rep["insert_tilt_series"] = {
        "workload": f"insert_central_slices_3d of {b} CTF-weighted 256^2 slices of a +-60 deg single-axis tilt series "
                    "(random in-plane angles) into 256^3 + weights (h2h)", **{k + "_ms": v for k, v in tilt_ms.items()}}
    log(f"tilt-series insertion: {tilt_ms['model_plan']:.3f} ms (model plan), "
        f"{tilt_ms['pose_adaptive_plan']:.3f} ms (pose-adaptive plan)")
    del tv, tw, tinv

    # Isotropic CTF of a reconstructed 256^3 rfft volume (h2h): the volume multiplied by CTF(|f|) in place.
    spec = torch.randn((1, n, n, n // 2 + 1), dtype=torch.complex64, device=dev)
    ciso = ns.CTFIsotropic(1.0, 1.5, 300, 0.07, 2.7)
    t = timed(lambda: ns.ctf_isotropic("h2h", spec, spec, (1, n, n, n), ciso))
    nbytes = 2 * spec.numel() * 8
    rep["ctf_isotropic_volume"] = {
        "workload": f"ctf_isotropic of a {n}^3 c32 rfft volume (h2h) in place, CTFIsotropic<f32>",
        "avg_ms": t * 1e3, "algorithmic_bytes": nbytes, "achieved_GBs": nbytes / t / 1e9,
        "frac_hbm_peak": nbytes / t / 1e9 / HBM_PEAK_GBS}
    log(f"ctf isotropic {n}^3: {t * 1e3:.3f} ms, {nbytes / t / 1e9:.0f} GB/s")
    del spec

    # Cubic B-spline prefilter of a 256^3 f32 volume in place (before CUBIC_BSPLINE interpolation): three passes
    # (x, y, z), each reading and writing the volume once.
    vol = torch.randn((1, n, n, n), device=dev, dtype=torch.float32)
    t = timed(lambda: nx.cubic_bspline_prefilter(vol, vol))
    nbytes = 3 * 2 * vol.numel() * 4
    rep["bspline_prefilter"] = {
        "workload": f"cubic_bspline_prefilter of a {n}^3 f32 volume in place (x, y, z passes)",
        "avg_ms": t * 1e3, "algorithmic_bytes": nbytes, "achieved_GBs": nbytes / t / 1e9,
        "frac_hbm_peak": nbytes / t / 1e9 / HBM_PEAK_GBS}
    log(f"bspline prefilter: {t * 1e3:.3f} ms, {nbytes / t / 1e9:.0f} GB/s")

    # Gridding correction of the reconstructed 256^3 real volume in place (divided by sinc^2), and the h2hc remap of
    # the 256^3 rfft volume (out of place): one read and one write of the volume each.
    t = timed(lambda: nx.fourier_interpolation_correction(vol, vol))
    nbytes = 2 * vol.numel() * 4
    rep["gridding_correction"] = {
        "workload": f"fourier_interpolation_correction of a {n}^3 f32 volume in place (LINEAR, post-correction)",
        "avg_ms": t * 1e3, "algorithmic_bytes": nbytes, "achieved_GBs": nbytes / t / 1e9,
        "frac_hbm_peak": nbytes / t / 1e9 / HBM_PEAK_GBS}
    log(f"gridding correction: {t * 1e3:.3f} ms, {nbytes / t / 1e9:.0f} GB/s")
    del vol
    spec = torch.randn((1, n, n, n // 2 + 1), dtype=torch.complex64, device=dev)
    spec_c = torch.empty_like(spec)
    t = timed(lambda: nx.remap("h2hc", spec, spec_c, (1, n, n, n)))
    nbytes = 2 * spec.numel() * 8
    rep["remap_volume"] = {
        "workload": f"remap h2hc of a {n}^3 c32 rfft volume (out of place)",
        "avg_ms": t * 1e3, "algorithmic_bytes": nbytes, "achieved_GBs": nbytes / t / 1e9,
        "frac_hbm_peak": nbytes / t / 1e9 / HBM_PEAK_GBS}
    log(f"remap {n}^3: {t * 1e3:.3f} ms, {nbytes / t / 1e9:.0f} GB/s")
    del spec, spec_c

    # The standalone phase shift of 4096 extracted 256^2 slices (h2h) in place, one shift per slice.
    sl = torch.randn((4096, 1, n, n // 2 + 1), dtype=torch.complex64, device=dev)
    sh = torch.from_numpy(np.random.default_rng(12).uniform(-8, 8, (4096, 2)).astype(np.float32)).to(dev)
    t = timed(lambda: nx.phase_shift_2d("h2h", sl, sl, (4096, 1, n, n), sh))
    nbytes = 2 * sl.numel() * 8 + sh.numel() * 4
    rep["phase_shift_slices"] = {
        "workload": f"phase_shift_2d of 4096 {n}^2 rfft slices (h2h) in place, one shift per slice",
        "avg_ms": t * 1e3, "algorithmic_bytes": nbytes, "achieved_GBs": nbytes / t / 1e9,
        "frac_hbm_peak": nbytes / t / 1e9 / HBM_PEAK_GBS}
    log(f"phase shift 4096 slices: {t * 1e3:.3f} ms, {nbytes / t / 1e9:.0f} GB/s")
    del sl, sh

    # FFTs on either side of the path (rocFFT plans cached as in noa): the c2r of the reconstructed 256^3 rfft
    # volume, and the r2c of a stack of 1024 real 256^2 images into "h" slices.
    import noa_amd.fft as nf
    spec = torch.randn((1, n, n, n // 2 + 1), dtype=torch.complex64, device=dev)
    real = torch.empty((1, n, n, n), dtype=torch.float32, device=dev)
    t = timed(lambda: nf.c2r(spec, real))
    nbytes = spec.numel() * 8 + real.numel() * 4
    rep["fft_c2r_volume"] = {
        "workload": f"fft::c2r of a {n}^3 volume (c32 rfft -> f32), norm FORWARD",
        "avg_ms": t * 1e3, "algorithmic_bytes": nbytes, "achieved_GBs": nbytes / t / 1e9,
        "frac_hbm_peak": nbytes / t / 1e9 / HBM_PEAK_GBS}
    log(f"fft c2r {n}^3: {t * 1e3:.3f} ms, {nbytes / t / 1e9:.0f} GB/s")
    del spec, real
    imgs = torch.randn((1024, 1, n, n), dtype=torch.float32, device=dev)
    out = torch.empty((1024, 1, n, n // 2 + 1), dtype=torch.complex64, device=dev)
    t = timed(lambda: nf.r2c(imgs, out))
    nbytes = imgs.numel() * 4 + out.numel() * 8
    rep["fft_r2c_slices"] = {
        "workload": f"fft::r2c of 1024 real {n}^2 images (f32 -> c32 rfft), norm FORWARD (1/N fused in the transform)",
        "avg_ms": t * 1e3, "algorithmic_bytes": nbytes, "achieved_GBs": nbytes / t / 1e9,
        "frac_hbm_peak": nbytes / t / 1e9 / HBM_PEAK_GBS, "slices_per_s": 1024 / t}
    log(f"fft r2c 1024 x {n}^2: {t * 1e3:.3f} ms, {nbytes / t / 1e9:.0f} GB/s")

    # MRC IO: a stack of 1024 256^2 images stored as I16 (the usual raw-data mode), written from and read back
    # into f32 device memory (chunked through pinned buffers, decoded and encoded on the GPU). The file sits in
    # the page cache after the write, so the read rate is host memory + PCIe, not a disk's.
    import tempfile
    import noa_amd.io as nio
    stack = torch.round(imgs * 100).contiguous()
    del out
    with tempfile.TemporaryDirectory() as tmp:
        path = os.path.join(tmp, "stack.mrc")
        t0 = time.perf_counter()
        nio.write_image(stack, path, spacing=(1.0, 1.0, 1.0), dtype="I16")
        t_w = time.perf_counter() - t0
        dst = torch.empty_like(stack)
        nio.read_image(path, output=dst)
        t0 = time.perf_counter()
        nio.read_image(path, output=dst)
        t_r = time.perf_counter() - t0
        ok = bool(torch.equal(dst, torch.clamp(stack, -32768, 32767)))
    fbytes = stack.numel() * 2
    rep["mrc_io"] = {
        "workload": f"1024 x {n}^2 f32 device images <-> MRC mode 1 (I16) file, page-cached",
        "read_ms": t_r * 1e3, "write_ms": t_w * 1e3, "file_bytes": fbytes,
        "read_file_GBs": fbytes / t_r / 1e9, "write_file_GBs": fbytes / t_w / 1e9, "round_trip_exact": ok}
    log(f"mrc read {t_r * 1e3:.1f} ms ({fbytes / t_r / 1e9:.1f} GB/s of file), write {t_w * 1e3:.1f} ms")
    del imgs, stack, dst
    return rep


def _qps_list(text):
    return [q if q == "max" else float(q) for q in str(text).split(",") if q]


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=10)
    ap.add_argument("--warmup", type=int, default=2)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--n-insert", type=int, default=10_000)
    ap.add_argument("--n-extract", type=int, default=4096)
    ap.add_argument("--probe", action="store_true", help="one launch of each operator, no timing (counter runs)")
    ap.add_argument("--probe-extract", default="bricks", help="extraction layouts of --probe (linear,bricks,tiles)")
    ap.add_argument("--probe-insert", default="wave", help="insertion kernels of --probe (wave,slab)")
    ap.add_argument("--serve-qps", default="200,1000,3000,max",
                    help="offered loads of the serving sweep (requests/s, comma-separated; max = all at once)")
    ap.add_argument("--serve-requests", type=int, default=400, help="requests in the serving run (0: skip)")
    ap.add_argument("--serve-only", action="store_true", help="only the serving run")
    ap.add_argument("--no-neighbours", action="store_true",
                    help="skip the CTF prologue and virtual-volume timings (not part of the step)")
    ap.add_argument("--no-tune", action="store_true", help="skip the launch autotuner (library defaults)")
    ap.add_argument("--precision", action="store_true",
                    help="FP32/FP16/BF16 volume storage for the 256^3 extraction: error against the FP64 oracle")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only (got --gpus {args.gpus}); the multi-GPU path is not built.",
              file=sys.stderr)
        sys.exit(2)

    import torch
    import noa_amd.xform as nx
    from noa_amd import workloads

    dev = torch.device("cuda:0")
    if args.serve_only:
        print(json.dumps(serving_report(torch, dev, args.serve_requests, _qps_list(args.serve_qps))), flush=True)
        return
    log("generating inputs ...")
    ext = workloads.extract_256(dev, b=args.n_extract)
    if args.precision:
        print(json.dumps(precision_report(ext, nx, torch)), flush=True)
        return
    ins = workloads.insert_256(dev, b=args.n_insert, keep_raw=not args.probe)
    n = 256
    out = torch.empty((args.n_extract, 1, n, n // 2 + 1), dtype=torch.complex64, device=dev)
    vol = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.complex64, device=dev)
    wvol = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.float32, device=dev)
    torch.cuda.synchronize()

    shifts = torch.from_numpy(ext.shifts).to(dev)

    def extract():
        # extract_central_slices_3d then phase_shift_2d of the slices by their in-plane shifts, fused.
        nx.extract_central_slices_3d_shifted("hc2hc", ext.volume, None, ext.volume_shape, out, None, ext.slice_shape,
                                             None, ext.rotations, shifts=shifts)

    def insert():
        nx.insert_central_slices_3d("h2h", ins.slices, ins.weights, ins.slice_shape, vol, wvol, ins.volume_shape,
                                    None, ins.inv_rotations)

    if args.probe:
        # One launch of each operator and a device copy of known size (1 GiB read + 1 GiB written), for hardware
        # counter runs: the copy calibrates FETCH_SIZE / WRITE_SIZE against known bytes.
        src = torch.empty(1 << 28, dtype=torch.float32, device=dev).normal_()
        dst = torch.empty_like(src)
        torch.cuda.synchronize()
        dst.copy_(src)
        # One launch per requested variant (comma-separated), in order.
        for layout in args.probe_extract.split(","):
            os.environ["NOA_HIP_EXTRACT_LAYOUT"] = layout
            extract()
            torch.cuda.synchronize()
        for kernel in args.probe_insert.split(","):
            os.environ["NOA_HIP_INSERT_KERNEL"] = kernel
            insert()
            torch.cuda.synchronize()
        log(f"probe done: copy 1 GiB, extract ({args.probe_extract}), insert ({args.probe_insert})")
        return

    tuning = None
    if not args.no_tune:
        # The launch tuning of both operators on this workload (every candidate gives the same result bits or, for
        # insertion, results within the kernels' stated tolerance; only the work decomposition changes). Only the
        # kernel / layout is tuned: the other knobs (work-item sizes, item order) measured within noise of their
        # defaults, and the counter summaries under profiles/ describe the defaults.
        from noa_amd import abi, autotune
        log("autotune ...")
        ek = {"box": n, "remap": abi.HC2HC, "interp": 1, "dtype": abi.C32}
        ik = {"box": n, "remap": abi.H2H, "interp": 1, "dtype": abi.C32}
        be = autotune.tune("extract", extract, key=ek, reps=3, log=log,
                           candidates=[(1, 0), (2, 0), (3, 128)])
        bi = autotune.tune("insert", insert, key=ik, reps=3, log=log,
                           candidates=[(1, 256), (2, 512)])
        tuning = {"extract": {"layout": {1: "row-major gather", 2: "block-copy gather", 3: "LDS tiles"}[be.values[0]],
                              "tile_pairs": be.values[1], "ms": be.ms},
                  "insert": {"kernel": {1: "one-wave", 2: "slab"}[bi.values[0]], "slices_per_item": bi.values[1],
                             "item_order": {0: "by expected work", 2: "XCD-aware"}[bi.values[3]], "ms": bi.ms}}
        vol.zero_()
        wvol.zero_()

    log("warmup ...")
    for _ in range(args.warmup):
        extract()
        insert()
    torch.cuda.synchronize()

    # K steps bracketed by synchronisations; HIP events on the launch stream time each operator inside them.
    marks = [[torch.cuda.Event(enable_timing=True) for _ in range(3)] for _ in range(args.steps)]
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for k in range(args.steps):
        marks[k][0].record()
        extract()
        marks[k][1].record()
        insert()
        marks[k][2].record()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    durations = {"extract": [m[0].elapsed_time(m[1]) * 1e-3 for m in marks],
                 "insert": [m[1].elapsed_time(m[2]) * 1e-3 for m in marks]}
    ms_per_step = wall / args.steps * 1e3
    slices_per_step = args.n_extract + args.n_insert
    value = slices_per_step / (wall / args.steps)

    kernels = {}
    for name, nbytes, nsl in (("extract", algorithmic_bytes_extract(args.n_extract, n), args.n_extract),
                              ("insert", algorithmic_bytes_insert(args.n_insert, n), args.n_insert)):
        avg = statistics.mean(durations[name])
        gbs = nbytes / avg / 1e9
        kernels[name] = {"avg_ms": avg * 1e3, "algorithmic_bytes": nbytes, "achieved_GBs": gbs,
                         "frac_hbm_peak": gbs / HBM_PEAK_GBS, "slices_per_s": nsl / avg}
        log(f"{name}: {avg * 1e3:.3f} ms, {gbs:.0f} GB/s ({100 * gbs / HBM_PEAK_GBS:.1f}% of HBM peak), "
            f"{nsl / avg / 1e6:.2f} M slices/s")
    dom = max(kernels, key=lambda k: kernels[k]["avg_ms"])
    variant = {"insert": tuning["insert"]["kernel"] if tuning else "slab",
               "extract": tuning["extract"]["layout"] if tuning else "block-copy gather"}
    traffic, traffic_src = measured_traffic(dom, args.n_insert if dom == "insert" else args.n_extract, variant[dom])
    total_bytes = sum(k["algorithmic_bytes"] for k in kernels.values())
    total_time = sum(k["avg_ms"] for k in kernels.values()) * 1e-3

    result = {
        "metric": METRIC,
        "value": value,
        "unit": "slices/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_per_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {
            "workload": f"256^3 extract {args.n_extract} slices (hc, LINEAR) with their in-plane shifts applied by a "
                        f"fused phase_shift_2d + insert {args.n_insert} CTF-weighted slices with CTF^2 weights (h2h, "
                        "LINEAR, windowed sinc 1 voxel)",
            "volume": [256, 256, 256],
            "slices_per_step": slices_per_step,
            "combined_frac_hbm_peak": total_bytes / total_time / 1e9 / HBM_PEAK_GBS,
        },
        "roofline": {
            "bound": "hbm",
            "kernel": KERNELS[dom][variant[dom]],
            "achieved": kernels[dom]["achieved_GBs"],
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": kernels[dom]["frac_hbm_peak"],
            "traffic": traffic,
            "traffic_source": traffic_src,
        },
        "kernels": kernels,
        "tuning": tuning,
    }
    # The same step with the two operators on two streams (independent inputs and outputs): reported beside the
    # sequential step that `value` and the per-kernel times come from.
    side = torch.cuda.Stream(device=dev)
    main_stream = torch.cuda.current_stream(dev)

    def two_streams():
        side.wait_stream(main_stream)
        with torch.cuda.stream(side):
            extract()
        insert()
        main_stream.wait_stream(side)

    for _ in range(args.warmup):
        two_streams()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        two_streams()
    torch.cuda.synchronize()
    wall2 = time.perf_counter() - t0
    result["two_streams"] = {"ms_per_step": wall2 / args.steps * 1e3,
                             "slices_per_s": slices_per_step / (wall2 / args.steps),
                             "note": "extraction on a second stream, concurrent with the insertion; not `value`"}
    log(f"two streams: {wall2 / args.steps * 1e3:.3f} ms per step, "
        f"{slices_per_step / (wall2 / args.steps) / 1e6:.2f} M slices/s")
    if not args.no_neighbours:
        log("prologue / virtual volume ...")
        result["neighbours"] = neighbours_report(torch, dev, nx, ins, n)
    if not args.no_cpu_baseline:
        log("cpu baseline ...")
        result["cpu_baseline"] = cpu_baseline(ext, ins)
    if args.serve_requests > 0:
        log("serving ...")
        del ext, ins, out
        torch.cuda.empty_cache()
        result["serving"] = serving_report(torch, dev, args.serve_requests, _qps_list(args.serve_qps))
    print(json.dumps(result), flush=True)


if __name__ == "__main__":
    main()
