#!/usr/bin/env python
"""Throughput bench of the dexel dilation hot path on one MI355X.

Workload (one step): dilation by r=16 of a direct dexel volume on a
1024x1024 grid, z-extent 1024, Poisson(6) segments per column with
exponential (mean 40 dexel) gaps and lengths, endpoints stored as FP32 on the
device (predicates and endpoint arithmetic in FP64).  Inputs are resident in
HBM before the timed region; a step is one vo_morph_device() call (block
summaries, the one-pass dilation, output CSR assembly), synchronised.

Prints ONE JSON line (see the keys below).  `roofline` is computed for the
dominant kernel from its average duration over the timed steps, measured with
HIP events that the library records on its own stream around each kernel
(`pass1_ms` the summaries, `pass2_ms` the one-pass dilation); its byte count
is algorithmic: per column the input is read once (2*s_in*E + 8) and the
output written once (2*s_out*E + 8), with E = 4 bytes and 8 of offset.
`cpu_baseline` times the CPU oracle (the FP64 restatement of `ours`) on a
bounded crop of the same volume, on this host's cores.
"""

import argparse
import json
import math
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "dexel columns/s + % HBM peak, 1024² r=16 dilation; batched FP32 vs plain FP64"
HBM_PEAK_GBS = 8000.0


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def _crop(vol, crop):
    from voroffset_amd.volume import CompressedVolume
    cols = [vol.at(x, y) for y in range(crop) for x in range(crop)]
    return CompressedVolume.from_columns(crop, crop, cols, origin=vol.origin, extent=vol.extent,
                                         spacing=vol.spacing, padding=vol.padding)


def cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(vol, radius, threads, crop, crop1):
    """The oracle's `ours` (FP64 restatement, line-parallel with grain 10
    lines like the reference's dormant TBB path) on crop x crop of the
    workload (the whole volume when crop covers it) with `threads` threads,
    and single-threaded on crop1 x crop1.
    Also returns the full-volume mean pass-1 triple count m (for the byte
    figure)."""
    import oracle

    t = time.perf_counter()
    po = oracle.pass1(vol, radius, threads=threads)[0]
    m = float(np.diff(po).mean())
    log(f"oracle pass-1 count m={m:.3f} ({time.perf_counter() - t:.1f} s)")
    whole = crop >= max(vol.nx, vol.ny)
    sample = vol if whole else _crop(vol, crop)
    t = time.perf_counter()
    oracle.morph(sample, "dilation", radius, "ours", threads=threads)
    dt = time.perf_counter() - t
    single = _crop(vol, crop1)
    t = time.perf_counter()
    oracle.morph(single, "dilation", radius, "ours", threads=1)
    dt1 = time.perf_counter() - t
    return m, {"value": round(sample.ncols / dt, 1), "unit": "dexel columns/s", "cores": threads, "kind": "port",
               "sample": (f"the whole {vol.nx}x{vol.ny} volume" if whole else f"{crop}x{crop} crop of the same volume")
                         + f", oracle `ours` (FP64) dilation r={radius:g}, {threads} threads, {dt:.1f} s",
               "single_thread": {"value": round(single.ncols / dt1, 1), "cores": 1,
                                 "sample": f"{crop1}x{crop1} crop, 1 thread, {dt1:.1f} s"},
               "host_cpus": os.cpu_count(), "cpu_model": cpu_model(),
               "oracle": "the repository's FP64 CPU restatement of `ours` (oracle/vo_oracle.cpp), pinned by "
                         "closed forms, `ours` == `brute_force` on all four operations and the pass-1 envelope "
                         "identity; the reference itself cannot be compiled here (its core needs Eigen)"}


# -- precision report ----------------------------------------------------------
# A check item is one GPU result (FP32 storage) on a window, beside the FP64
# input it was computed from, cropped with enough margin that the window's
# columns see all the input they depend on (the radius, twice for closing and
# opening; a crop that reaches the grid border keeps that border).  The
# cpu_baseline leg runs the oracle on each crop and compares the window.

def _reach(op, r):
    k = int(math.floor(r))
    return 2 * k + 1 if op in ("closing", "opening") else k + 1


def window_item(label, vol, res, op, r, x0, y0, w):
    """A check item for the w x w window at (x0, y0) of `res` = op(vol)."""
    m = _reach(op, r)
    cx0, cy0 = max(0, x0 - m), max(0, y0 - m)
    cx1, cy1 = min(vol.nx, x0 + w + m), min(vol.ny, y0 + w + m)
    win = res.crop(x0, y0, w, w)
    return {"config": label, "op": op, "r": r, "input": vol.crop(cx0, cy0, cx1 - cx0, cy1 - cy0),
            "window": (x0 - cx0, y0 - cy0, w, w), "off": win.off, "z": win.z}


def whole_item(label, vol, res, op, r):
    return {"config": label, "op": op, "r": r, "input": vol, "window": (0, 0, vol.nx, vol.ny),
            "off": res.off, "z": res.z}


def direct_items(vol, windows=((500, 300), (131, 877)), w=24):
    """Config 3 (the bench volume): dilation and erosion at r = 16 and 64,
    closing at r = 16, FP32 storage through the host entry point."""
    from voroffset_amd.morpho import VoronoiMorphoHip

    hip = VoronoiMorphoHip("fp32")
    items = []
    try:
        for op, r in (("dilation", 16.0), ("dilation", 64.0), ("erosion", 16.0), ("erosion", 64.0),
                      ("closing", 16.0)):
            res, _, _ = hip.apply(op, vol, r)
            items += [window_item(f"direct {vol.nx}^2", vol, res, op, r, x, y, w) for x, y in windows]
    finally:
        hip.close()
    return items


def mesh_items():
    """Configs 1 and 2: the 32-sphere mesh (128 dexels, padding 8, dilation
    r = 4, whole volume) and the 2000-tube mesh (512 box, padding 16:
    dilation 10, erosion 3, opening / closing 5, on two windows), rasterized
    and processed on the GPU."""
    from voroffset_amd import mesh as M
    from voroffset_amd.morpho import VoronoiMorphoHip

    hip = VoronoiMorphoHip("fp32")
    items = []
    try:
        spheres = M.create_dexels(M.icosphere_union(32, level=3, seed=1), 1.0, 8, 128, ctx=hip.ctx)
        res, _, _ = hip.apply("dilation", spheres, 4.0)
        items.append(whole_item("spheres 128", spheres, res, "dilation", 4.0))
        tubes = M.create_dexels(M.prism_tubes(2000, box=512.0, seed=2), 1.0, 16, -1, ctx=hip.ctx)
        for op, r in (("dilation", 10.0), ("erosion", 3.0), ("opening", 5.0), ("closing", 5.0)):
            res, _, _ = hip.apply(op, tubes, r)
            items += [window_item("tubes 512", tubes, res, op, r, x, y, 32)
                      for x, y in ((tubes.nx // 2, tubes.ny // 3), (100, 380))]
    finally:
        hip.close()
    return items


def precision_report(items, threads):
    """Per config: the max endpoint error of the FP32-storage GPU results
    against the FP64 oracle on the FP64 input (so it includes the float32
    rounding of the input), columns compared, columns whose segment counts
    differ, and how many of those only differ by gaps narrower than 1e-5
    dexel, or by segments that narrow where such a gap is complemented
    (the rest are listed as unexplained)."""
    import oracle

    rep = {}
    for it in items:
        ro, rz = oracle.morph(it["input"], it["op"], it["r"], threads=threads)
        ref = it["input"].like(ro, rz).crop(*it["window"])
        la, lb = np.diff(it["off"]), np.diff(ref.off)
        bad = np.nonzero(la != lb)[0]
        same = np.nonzero((la == lb) & (la > 0))[0]
        err = 0.0
        if same.size:
            ia = np.concatenate([np.arange(it["off"][c], it["off"][c + 1]) for c in same])
            ib = np.concatenate([np.arange(ref.off[c], ref.off[c + 1]) for c in same])
            err = float(np.max(np.abs(it["z"][ia] - ref.z[ib])))

        def fused(z):
            out = []
            for k in range(0, len(z), 2):
                if out and z[k] - out[-1] < 1e-5:
                    out[-1] = max(out[-1], z[k + 1])
                else:
                    out.extend([z[k], z[k + 1]])
            return sum(1 for k in range(0, len(out), 2) if out[k + 1] - out[k] >= 1e-5)
        narrow = sum(1 for c in bad if fused(it["z"][it["off"][c]:it["off"][c + 1]]) ==
                     fused(ref.z[ref.off[c]:ref.off[c + 1]]))
        key = f'{it["config"]}: {it["op"]} r={it["r"]:g}'
        e = rep.setdefault(key, {"max_err": 0.0, "columns": 0, "count_mismatch": 0, "narrow_gap": 0,
                                 "unexplained": 0})
        e["max_err"] = max(e["max_err"], err)
        e["columns"] += int(la.size)
        e["count_mismatch"] += int(bad.size)
        e["narrow_gap"] += int(narrow)
        e["unexplained"] += int(bad.size - narrow)
    for e in rep.values():
        e["max_err"] = float(f'{e["max_err"]:.3g}')
    return rep


def _bucket(radius):
    r = int(radius)
    return 0 if r < 8 else 1 if r < 16 else 2 if r < 32 else 3 if r < 64 else 4


def run_device(ctx, vol, radius, precision, steps, warmup):
    from voroffset_amd import _native

    zlo, zhi = vol.z_range()
    shift = _native.storage_shift(zlo, zhi) if precision == "fp32" else 0.0
    dtype = np.float32 if precision == "fp32" else np.float64
    d_off = _native.DeviceArray(vol.off)
    d_z = _native.DeviceArray((vol.z - shift).astype(dtype))
    args = ("dilation", precision, radius, vol.nx, vol.ny, d_off.address, d_z.address, zlo - shift, zhi - shift)
    for _ in range(warmup):
        ctx.morph_device(*args)
    _native.synchronize()
    p1 = p2 = 0.0
    t0 = time.perf_counter()
    for _ in range(steps):
        _, count, (t1, t2) = ctx.morph_device(*args)
        p1 += t1
        p2 += t2
    _native.synchronize()
    dt = time.perf_counter() - t0
    d_off.free()
    d_z.free()
    return dt / steps, p1 / steps, p2 / steps, count


def takes_sweeps(radius):
    """Whether dilations by `radius` may take the two sweeps, whose shapes the
    autotuner picks (the one-pass form has nothing to tune)."""
    return bool(os.environ.get("VO_PASS1") or os.environ.get("VO_PASS2")) or radius < 6 or radius >= 256


def tune_context(ctx, lam, radii, side=256, seed=7):
    """Untimed: autotunes ctx's shapes for these radii on a side x side
    Poisson(lam) sample volume (FP32 storage)."""
    from voroffset_amd import _native, synth

    v = synth.poisson_columns(side, side, lam=lam, zmax=1024, seed=seed)
    zlo, zhi = v.z_range()
    shift = _native.storage_shift(zlo, zhi)
    d_off, d_z = _native.DeviceArray(v.off), _native.DeviceArray((v.z - shift).astype(np.float32))
    try:
        return ctx.autotune("fp32", v.nx, v.ny, d_off.address, d_z.address, radii, reps=3)
    finally:
        d_off.free()
        d_z.free()


def tune_batch(ctx, jobs, buckets, choices=(512, 768, 1024, 1536), reps=2):
    """Untimed: tunes the z-sweep events per slab of each radius bucket the
    batch uses on the batch itself (one bucket at a time, the others held),
    keeping the default where no choice is faster; returns the tuning."""
    import tempfile
    from voroffset_amd import _native

    def run():
        ctx.morph_batch_device("fp32", jobs)  # eager, then captured: timed replays
        ctx.morph_batch_device("fp32", jobs)
        _native.synchronize()
        t = time.perf_counter()
        for _ in range(reps):
            ctx.morph_batch_device("fp32", jobs)
        _native.synchronize()
        return (time.perf_counter() - t) / reps

    table = ctx.tuning()
    with tempfile.TemporaryDirectory() as tmp:
        path = os.path.join(tmp, "tuning")

        def load(tab):
            with open(path, "w") as f:
                f.write("voroffset_amd tuning 1\n" + "".join(f"{b} {e} {o}\n" for b, (e, o) in enumerate(tab)))
            ctx.tuning_load(path)
        best = run()
        for b in buckets:
            for e in choices:
                if e == table[b][0]:
                    continue
                trial = list(table)
                trial[b] = (e, table[b][1])
                load(trial)
                t = run()
                if t < best * 0.99:
                    best, table = t, trial
        load(table)
    return table


def batched_leg(n_volumes, steps, warmup, seed=4321, tune=True):
    """The uneven batch: n volumes, side log-uniform in [64, 512], Poisson(lambda
    ~ U[2, 10]) segments per column, r ~ U[2, 32], ops uniform over dilation /
    erosion / closing / opening.  Batched FP32 (one vo_morph_batch_device call
    for all volumes) against plain per-volume FP64 calls, inputs resident in
    HBM, each timed over whole batches."""
    from voroffset_amd import _native, synth

    specs = synth.batch_specs(n_volumes, seed=seed)
    keep, jobs32, jobs64, cols = [], [], [], 0
    for sp in specs:
        v = synth.poisson_columns(sp["side"], sp["side"], lam=sp["lam"], zmax=1024, seed=sp["seed"])
        zlo, zhi = v.z_range()
        shift = _native.storage_shift(zlo, zhi)
        d_off = _native.DeviceArray(v.off)
        d32 = _native.DeviceArray((v.z - shift).astype(np.float32))
        d64 = _native.DeviceArray(v.z)
        keep += [d_off, d32, d64]
        jobs32.append((sp["op"], sp["radius"], v.nx, v.ny, d_off.address, d32.address, zlo - shift, zhi - shift))
        jobs64.append((sp["op"], sp["radius"], v.nx, v.ny, d_off.address, d64.address, zlo, zhi))
        cols += v.ncols
    ctx = _native.Context(0)
    tuned = None
    if tune:
        buckets = sorted({_bucket(sp["radius"]) for sp in specs})
        tuned = tune_batch(ctx, jobs32, buckets)
        log(f"batch tuning (events per slab, list capacity per radius bucket): {tuned}")
    for _ in range(warmup):
        ctx.morph_batch_device("fp32", jobs32)
    _native.synchronize()
    t = time.perf_counter()
    for _ in range(steps):
        ctx.morph_batch_device("fp32", jobs32)
    _native.synchronize()
    tb = (time.perf_counter() - t) / steps
    alone = ctx.last_batch_alone()

    def plain():
        for (op, r, nx, ny, off, z, zlo, zhi) in jobs64:
            ctx.morph_device(op, "fp64", r, nx, ny, off, z, zlo, zhi)
    for _ in range(warmup):
        plain()
    _native.synchronize()
    t = time.perf_counter()
    for _ in range(steps):
        plain()
    _native.synchronize()
    tp = (time.perf_counter() - t) / steps
    # results of four sampled volumes of side <= 256 for the precision report
    from voroffset_amd.volume import CompressedVolume
    outs, _ = ctx.morph_batch_device("fp32", jobs32)
    rng = np.random.default_rng(seed)
    small = [k for k, sp in enumerate(specs) if sp["side"] <= 256]
    items = []
    for k in sorted(rng.choice(small, min(4, len(small)), replace=False).tolist()):
        v, cnt = outs[k]
        sp = specs[k]
        src = synth.poisson_columns(sp["side"], sp["side"], lam=sp["lam"], zmax=1024, seed=sp["seed"])
        zlo, zhi = src.z_range()
        shift = _native.storage_shift(zlo, zhi)
        res = src.like(_native.to_host(v.offsets, np.int64, v.nx * v.ny + 1),
                       _native.to_host(v.z, np.float32, cnt).astype(np.float64) + shift)
        items.append(whole_item(f"batch of {n_volumes}", src, res, sp["op"], sp["radius"]))
    ctx.close()
    for d in keep:
        d.free()
    log(f"batched: {n_volumes} volumes, {cols} columns; fp32 batch {tb * 1e3:.2f} ms, plain fp64 {tp * 1e3:.2f} ms "
        f"({tp / tb:.2f}x), {alone} volumes redone alone")
    return {"workload": f"{n_volumes} volumes, side log-uniform [64, 512], Poisson(U[2,10]) segments/column, "
                        f"r U[2,32], ops uniform over dilation/erosion/closing/opening, seed {seed}",
            "columns": cols, "batched_fp32": {"value": round(cols / tb, 1), "ms_per_batch": round(tb * 1e3, 3)},
            "plain_fp64": {"value": round(cols / tp, 1), "ms_per_batch": round(tp * 1e3, 3)},
            "batched_over_plain": round(tp / tb, 3), "volumes_redone_alone": alone,
            "tuning": tuned}, items


def served_leg(rate, n_requests, pool, seed=99, tune=True):
    """Served form: `pool` resident volumes (side log-uniform in [128, 2048],
    Poisson(8) segments per column), Poisson arrivals at `rate` per second of
    n_requests mixed jobs (op uniform, r ~ U[2, 48]); FP32 storage, HBM-budget
    admission, batches drained first-come first-served.  The achieved rate is
    reported beside the rate the Poisson draw realised over its arrival span,
    and the capacity is the same requests queued at once and drained."""
    from voroffset_amd import serve, synth

    rng = np.random.default_rng(seed)
    sides = np.round(np.exp(rng.uniform(math.log(128), math.log(2048), pool))).astype(int)
    srv = serve.MorphoServer("fp32", hbm_budget=64 << 30, max_batch=64)
    try:
        if tune:
            tune_context(srv.ctx, 8, [4.0, 12.0, 24.0, 40.0])
        handles, cols = [], {}
        for i, side in enumerate(sides):
            v = synth.poisson_columns(int(side), int(side), lam=8, zmax=1024, seed=seed * 1000 + i)
            h = srv.put(v)
            handles.append(h)
            cols[h] = v.ncols
        for h in handles:  # warm the workspace with the largest jobs
            srv.submit(h, "closing", 48.0)
        while srv.queue:
            for req in srv.step():
                srv.drop(req.result)
        srv.batches.clear()
        t = time.perf_counter()
        done = serve.simulate(srv, handles, rate, n_requests, seed=seed)
        span = max(r.done for r in done) - min(r.arrival for r in done)
        arr = sorted(r.arrival for r in done)
        offered = (len(arr) - 1) / max(arr[-1] - arr[0], 1e-9)  # the rate the Poisson draw realised
        rep = serve.latency_report(done)
        total = sum(cols[r.handle] for r in done)
        nb = len(srv.batches)
        # capacity: the same requests all queued at once, drained back to back
        cap = serve.simulate(srv, handles, rate, n_requests, seed=seed, saturate=True)
        cap_span = max(r.done for r in cap) - min(r.arrival for r in cap)
        # two results on the largest resident volume for the precision report
        big = int(np.argmax(sides))
        src = synth.poisson_columns(int(sides[big]), int(sides[big]), lam=8, zmax=1024, seed=seed * 1000 + big)
        items = []
        for op, r in (("closing", 48.0), ("dilation", 30.5)):
            req = srv.submit(handles[big], op, r)
            while srv.queue:
                srv.step()
            res = srv.get(req.result, src)
            srv.drop(req.result)
            s0 = src.nx
            items += [window_item(f"served {s0}^2", src, res, op, r, x, y, 24) for x, y in ((s0 // 2, s0 // 3),
                                                                                         (s0 - 24, 0))]
        rep.update({"workload": f"{pool} resident volumes, side log-uniform [128, 2048], Poisson(8) segments/column; "
                                f"{n_requests} requests, Poisson arrivals at {rate:g}/s, op uniform, r U[2,48]",
                    "offered_rate_per_s": rate, "offered_realised_per_s": round(offered, 2),
                    "columns_per_s": round(total / span, 1),
                    "requests_per_s": round(len(done) / span, 2), "batches": nb,
                    "mean_batch": round(float(np.mean([b for b, _ in srv.batches[:nb]])), 2),
                    "capacity_requests_per_s": round(len(cap) / cap_span, 2),
                    "wall_s": round(time.perf_counter() - t, 3)})
        log(f"served: p50 {rep['p50_ms']} ms, p99 {rep['p99_ms']} ms, {rep['requests_per_s']} req/s "
            f"(arrivals realised {offered:.1f}/s), {rep['columns_per_s']:.3g} columns/s, {rep['batches']} batches; "
            f"capacity {rep['capacity_requests_per_s']} req/s")
        return rep, items
    finally:
        srv.close()


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--side", type=int, default=1024)
    ap.add_argument("--radius", type=float, default=16.0)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--cpu-threads", type=int, default=min(16, os.cpu_count() or 1))
    ap.add_argument("--cpu-crop", type=int, default=1024, help="crop side of the all-threads CPU sample (1024: the whole volume)")
    ap.add_argument("--cpu-crop1", type=int, default=192, help="crop side of the single-thread CPU sample")
    ap.add_argument("--no-fp64", action="store_true", help="skip the plain FP64 leg (counter runs)")
    ap.add_argument("--no-tune", action="store_true", help="keep the default shapes (skip the autotuner)")
    ap.add_argument("--no-precision", action="store_true", help="skip the precision report (oracle checks)")
    ap.add_argument("--batch-volumes", type=int, default=256, help="volumes of the batched leg (0: skip it)")
    # 1000 requests (5 s of arrivals at 200/s): the achieved rate is requests
    # over first arrival to last completion, so the last requests' latency
    # weighs 5x less than over 200
    ap.add_argument("--serve-requests", type=int, default=1000, help="requests of the served leg (0: skip it)")
    ap.add_argument("--serve-rate", type=float, default=200.0, help="offered requests per second")
    ap.add_argument("--serve-pool", type=int, default=16, help="resident volumes of the served leg")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py runs on exactly one GPU (this build has no multi-GPU path); got --gpus {args.gpus}",
              file=sys.stderr)
        sys.exit(2)

    from voroffset_amd import _native, synth

    R, side = args.radius, args.side
    vol = synth.poisson_columns(side, side, lam=6, zmax=1024, seed=1234)
    ncols = vol.ncols
    ctx = _native.Context(0)
    tuned = None
    if not args.no_tune and takes_sweeps(R):  # untimed: the autotuner picks the shapes for this radius on the workload itself
        zlo, zhi = vol.z_range()
        shift = _native.storage_shift(zlo, zhi)
        d_off, d_z = _native.DeviceArray(vol.off), _native.DeviceArray((vol.z - shift).astype(np.float32))
        t = time.perf_counter()
        table = ctx.autotune("fp32", vol.nx, vol.ny, d_off.address, d_z.address, [R], reps=3)
        d_off.free()
        d_z.free()
        tuned = {"events_per_slab": table[_bucket(R)][0], "gather_list_capacity": table[_bucket(R)][1]}
        log(f"autotune ({time.perf_counter() - t:.1f} s): {tuned}")

    step_s, p1_ms, p2_ms, count = run_device(ctx, vol, R, "fp32", args.steps, args.warmup)
    fallback = ctx.last_stats()[1]
    log(f"fp32: {step_s * 1e3:.3f} ms/step, pass1 {p1_ms:.3f} ms, pass2 {p2_ms:.3f} ms, "
        f"{fallback} tiles computed again")
    plain = None
    if not args.no_fp64:
        f64_s, f64_p1, f64_p2, _ = run_device(ctx, vol, R, "fp64", max(3, args.steps // 4), 1)
        log(f"fp64: {f64_s * 1e3:.3f} ms/step, pass1 {f64_p1:.3f} ms, pass2 {f64_p2:.3f} ms")
        plain = {"value": round(ncols / f64_s, 1), "ms_per_step": round(f64_s * 1e3, 4),
                 "pass1_ms": round(f64_p1, 4), "pass2_ms": round(f64_p2, 4)}

    # a batch in the two sweeps is tuned on its own uneven volumes (shapes tuned
    # on one uniform sample made it slower: 39.3 ms against 35.6 ms untuned);
    # the served leg keeps the default shapes
    items = []
    batched = None
    if args.batch_volumes > 0:
        # untimed batches: the first runs eagerly, the second captures the
        # program into a HIP graph, and after some more its tables' upload
        # is at its steady speed (14.3 -> 13.5 ms); the timed ones replay it
        batched, more = batched_leg(args.batch_volumes, max(2, args.steps // 5), 16,
                                    tune=not args.no_tune and takes_sweeps(16.0))
        items += more

    served = None
    if args.serve_requests > 0:
        served, more = served_leg(args.serve_rate, args.serve_requests, args.serve_pool, tune=False)
        items += more

    m, cpu, precision = (None, None, None)
    if not args.no_cpu:
        m, cpu = cpu_baseline(vol, R, args.cpu_threads, args.cpu_crop, args.cpu_crop1)
        log(f"cpu baseline: {cpu['value']:.3g} columns/s")
        if not args.no_precision:  # the oracle as the checker of GPU results computed above
            t = time.perf_counter()
            precision = precision_report(direct_items(vol) + mesh_items() + items, args.cpu_threads)
            log(f"precision report ({time.perf_counter() - t:.1f} s): "
                f"max err {max(e['max_err'] for e in precision.values()):.3g}, "
                f"unexplained count mismatches {sum(e['unexplained'] for e in precision.values())}")

    E = 4
    s_in = vol.num_segments() / ncols
    s_out = count / 2 / ncols
    roofline = None
    if not takes_sweeps(R):  # the one-pass form: summaries, then the dilation
        b = ncols * ((2 * s_in * E + 8) + (2 * s_out * E + 8))
        name, ms = "direct", p2_ms
        achieved = b / (ms * 1e-3) / 1e9
        # the instantiation the timed steps ran (FP32 storage, this radius);
        # counters measured on another one are not attached
        # (one wavefront a tile: the default grid's 16384 tiles)
        inst = f"direct_kernel<float, 3, {'true' if int(R) <= 9 else 'false'}, 1>"
        traffic, tnote = None, "no counter profile of this kernel in profiles/"
        tpath = os.path.join(ROOT, "profiles", f"traffic_{name}_1024_r16.json")
        if os.path.exists(tpath):
            prof = json.load(open(tpath))
            if prof.get("kernel") == inst:
                traffic, tnote = prof.get("hbm_bytes_per_launch"), os.path.relpath(tpath, ROOT)
            else:
                tnote = f"{os.path.relpath(tpath, ROOT)} profiles {prof.get('kernel')}, not the timed {inst}"
        roofline = {"bound": "hbm", "achieved": round(achieved, 2), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                    "frac": round(achieved / HBM_PEAK_GBS, 5), "traffic": traffic, "traffic_source": tnote,
                    "kernel": inst, "kernel_ms": round(ms, 4), "algorithmic_bytes": int(b),
                    "step_algorithmic_GBs": round(b / step_s / 1e9, 2)}

    out = {
        "metric": METRIC,
        "value": round(ncols / step_s, 1),
        "unit": "dexel columns/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(step_s * 1e3, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic",
        "config": {"workload": f"direct dexel volume {side}x{side}, z 1024, Poisson(6) segments/column, "
                               f"Exp(40) gaps and lengths, dilation r={R:g}, one volume per launch",
                   "grid": [side, side], "radius": R, "storage": "fp32", "op": "dilation",
                   "pass1_ms": round(p1_ms, 4), "pass2_ms": round(p2_ms, 4),
                   "plain_fp64": plain, "tiles_computed_again": fallback, "autotuned": tuned, "batched": batched,
                   "served": served,
                   "s_in": round(s_in, 4), "s_out": round(s_out, 4), "m_oracle": m,
                   "precision": precision},
        "roofline": roofline,
        "cpu_baseline": cpu,
    }
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
