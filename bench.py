#!/usr/bin/env python3
"""Benchmark of the GPU `path` integrator on the large-mesh stress scene.

Workload (default): 1920x1080, 64 spp, max depth 16, a 2048x2048-vertex fBm
terrain (8.38M triangles) plus 256 UV spheres of 2,116 triangles with GGX
conductor / rough dielectric / Disney materials, a constant environment and
a small distant spherical "sun" emitter.  One step = one full render of that
frame.  Prints one JSON line.

The CPU baseline is the oracle (the CPU restatement of the reference's
integrator, its own binned-SAH BVH, OpenMP over tiles) timed on an even
subsample of the same frame's tiles at full spp.

`--copy-probe MIB` instead runs a plain device-to-device copy of MIB MiB a
few times; its FETCH_SIZE / WRITE_SIZE counter readings calibrate the
counters that give the traversal kernel's HBM traffic.
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "samples/s at equal relMSE, guided vs plain GPU path; p50/p99 render latency"
HBM_PEAK_GBS = 8000.0
TRACE_BYTES_PER_RAY = 52  # ray read 32 B + hit write 20 B per closest-hit query


def parse():
    p = argparse.ArgumentParser()
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=3)
    p.add_argument("--warmup", type=int, default=2)
    p.add_argument("--config", default="large_mesh", choices=["large_mesh", "many_balls", "volume_box"])
    p.add_argument("--spp", type=int, default=None)
    p.add_argument("--cpu-seconds", type=float, default=15.0, help="target CPU-baseline sample duration")
    p.add_argument("--no-cpu", action="store_true")
    p.add_argument("--grid", type=int, default=2048)
    p.add_argument("--copy-probe", type=int, default=0, metavar="MIB")
    p.add_argument("--no-guiding", action="store_true", help="skip the guided-vs-plain measurement")
    p.add_argument("--summarize-counters", nargs="+", metavar="PMC_DIR",
                   help="print per-kernel counter sums of rocprofv3 --pmc output directories and exit")
    p.add_argument("--summarize-overlap", metavar="TRACE",
                   help="print how much kernels of different streams overlap in a rocprofv3 kernel trace and exit")
    p.add_argument("--serving-only", action="store_true", help="only the serving stream measurement; prints its record")
    p.add_argument("--guiding-only", action="store_true",
                   help="only the guided-vs-plain measurement (quirks off); prints its record")
    p.add_argument("--unsorted", action="store_true", help="shade with one kernel (no material sort)")
    p.add_argument("--no-autotune", action="store_true", help="keep the default launch configuration")
    p.add_argument("--launch", default=None, metavar="SLOTS,BPC,TPC",
                   help="fixed launch configuration (path slots, shade blocks per CU, trace blocks per CU); no autotune")
    p.add_argument("--builder", choices=["host", "device"], default="device", help="BVH builder")
    p.add_argument("--no-serving", action="store_true", help="skip the serving-latency measurement")
    p.add_argument("--guide-scale", type=float, default=1.0, help="image scale of the guiding workload")
    p.add_argument("--serve-requests", type=int, default=40)
    p.add_argument("--summarize", nargs="+", metavar="DIR",
                   help="TRACE [FETCH WRITE COPY_FETCH COPY_WRITE PMC_JSON]: print a text summary of rocprofv3 "
                        "csv output directories (the kernel trace alone, or with the traffic counters); "
                        "PMC_JSON: the bench line of "
                        "the counter runs (their segment count gives the traffic per ray)")
    return p.parse_args()


def _csv_rows(d, suffix):
    import csv
    import glob

    rows = []
    for f in sorted(glob.glob(os.path.join(d, "*" + suffix))):
        rows += list(csv.DictReader(open(f)))
    return rows


def _short(name):
    return name.replace("(anonymous namespace)::", "").split("(")[0].replace("void ", "")


TRAFFIC_TAG = "TRAFFIC k_extend bytes_per_ray="
PROFILE_SUMMARY = os.path.join(os.path.dirname(os.path.abspath(__file__)), "profiles", "k_extend_large_mesh.txt")


def summarize(dirs, copy_mib=1024):
    """Kernel-trace statistics plus FETCH_SIZE / WRITE_SIZE per dispatch,
    scaled by the readings of the plain copy of `copy_mib` MiB, and the
    closest-hit kernel's traffic per traced ray."""
    if len(dirs) not in (1, 6):
        raise SystemExit("--summarize takes TRACE, or TRACE FETCH WRITE COPY_FETCH COPY_WRITE PMC_JSON")
    trace = dirs[0]
    W = 44
    out = [f"{'kernel':{W}s} calls   total_ms    avg_us    min_us    max_us   vgpr  scratch"]
    stats = {}
    for r in _csv_rows(trace, "kernel_stats.csv"):
        stats[_short(r["Name"])] = r
    res = {}
    for r in _csv_rows(trace, "kernel_trace.csv"):
        res.setdefault(_short(r["Kernel_Name"]), (r["VGPR_Count"], r["Scratch_Size"]))
    for k, r in sorted(stats.items(), key=lambda kv: -float(kv[1]["TotalDurationNs"])):
        v, sc = res.get(k, ("?", "?"))
        out.append(f"{k[:W]:{W}s} {int(r['Calls']):6d} {float(r['TotalDurationNs']) / 1e6:10.2f} "
                   f"{float(r['AverageNs']) / 1e3:9.1f} {float(r['MinNs']) / 1e3:9.1f} {float(r['MaxNs']) / 1e3:9.1f} "
                   f"{v:>6s} {sc:>8s}")
    if len(dirs) == 1:
        return "\n".join(out)
    fetch, write, cfetch, cwrite, pmc_json = dirs[1:]

    def per_kernel(d):
        acc = {}
        for r in _csv_rows(d, "counter_collection.csv"):
            acc.setdefault(_short(r["Kernel_Name"]), []).append(float(r["Counter_Value"]))
        return acc

    cf, cw = per_kernel(cfetch), per_kernel(cwrite)
    copy_kib = copy_mib * 1024.0
    kf = [v for k, v in cf.items() if "copyBuffer" in k][0]
    kw = [v for k, v in cw.items() if "copyBuffer" in k][0]
    f_scale, w_scale = copy_kib / (sum(kf) / len(kf)), copy_kib / (sum(kw) / len(kw))
    out.append("")
    out.append(f"plain copy of {copy_mib} MiB: FETCH_SIZE {sum(kf) / len(kf):.0f} KiB, WRITE_SIZE "
               f"{sum(kw) / len(kw):.0f} KiB per dispatch -> scale factors fetch x{f_scale:.3f}, write x{w_scale:.3f}")
    out.append("")
    out.append(f"{'kernel':{W}s} dispatches  read_MB/launch  write_MB/launch  (scaled)")
    f, w = per_kernel(fetch), per_kernel(write)
    for k in sorted(f, key=lambda k: -sum(f[k])):
        if k not in w:
            continue
        rd = sum(f[k]) / len(f[k]) * f_scale * 1024 / 1e6
        wr = sum(w[k]) / len(w[k]) * w_scale * 1024 / 1e6
        out.append(f"{k[:W]:{W}s} {len(f[k]):10d} {rd:15.1f} {wr:16.1f}")
    ext = [k for k in f if k.split("<")[0].endswith("k_extend")]
    if ext and ext[0] in w:
        k = ext[0]
        line = json.loads(open(pmc_json).read().strip().splitlines()[-1])
        rays = line["stats"]["segments_per_step"] * line["steps"]
        total = (sum(f[k]) * f_scale + sum(w[k]) * w_scale) * 1024
        out.append("")
        out.append(f"k_extend: {rays:.0f} rays traced in the counter runs, {total / 1e9:.2f} GB read + written beyond L2")
        out.append(f"{TRAFFIC_TAG}{total / rays:.1f}")
    return "\n".join(out)


def summarize_counters(dirs):
    """Per-kernel sums of the counters in rocprofv3 --pmc output directories,
    with the derived rates the traversal analysis uses: VALU busy (SIMD cycles
    spent issuing VALU instructions over the SIMD cycles of the kernel), VALU
    lane utilisation (active lanes per VALU instruction / 64), the fractions
    of wave cycles spent waiting and issuing, L2 hit rate, the mean L1 -> L2
    read latency and the F16 MFMA work."""
    acc, launches = {}, {}
    for d in dirs:
        for r in _csv_rows(d, "counter_collection.csv"):
            k = _short(r["Kernel_Name"])
            c = acc.setdefault(k, {})
            c[r["Counter_Name"]] = c.get(r["Counter_Name"], 0.0) + float(r["Counter_Value"])
            launches.setdefault((d, k), set()).add(r["Dispatch_Id"])
    simds = xcc = None
    for d in dirs:
        for r in _csv_rows(d, "agent_info.csv"):
            if r.get("Name", "").startswith("gfx"):
                simds, xcc = int(r["Simd_Count"]), int(r["Num_Xcc"])
    out = []
    for k in sorted(acc):
        c = acc[k]
        n = max(len(v) for (d, kk), v in launches.items() if kk == k)
        out.append(f"{k}  ({n} dispatches per counter pass)")
        for name in sorted(c):
            out.append(f"  {name:32s} {c[name]:.4g}")
        dv = []
        if c.get("SQ_ACTIVE_INST_VALU") and "SQ_THREAD_CYCLES_VALU" in c:
            dv.append(f"VALU lane utilisation {c['SQ_THREAD_CYCLES_VALU'] / (64 * c['SQ_ACTIVE_INST_VALU']):.2f}")
        if simds and c.get("GRBM_GUI_ACTIVE") and "SQ_ACTIVE_INST_VALU" in c:
            # a wave64 VALU instruction holds its 16-lane SIMD for 4 cycles;
            # GRBM_GUI_ACTIVE counts the kernel's cycles once per XCC
            dv.append(f"VALU busy {4 * c['SQ_ACTIVE_INST_VALU'] / (simds * c['GRBM_GUI_ACTIVE'] / xcc):.2f} of SIMD cycles")
        if c.get("SQ_WAVE_CYCLES"):
            for name, lab in (("SQ_WAIT_ANY", "waiting"), ("SQ_ACTIVE_INST_ANY", "issuing")):
                if name in c:
                    dv.append(f"{lab} {c[name] / c['SQ_WAVE_CYCLES']:.2f} of wave cycles")
        if c.get("SQ_WAVES"):
            for name, lab in (("SQ_INSTS_VALU", "VALU"), ("SQ_INSTS_VMEM_RD", "VMEM rd"), ("SQ_INSTS_LDS", "LDS"),
                              ("SQ_INSTS_SALU", "SALU")):
                if name in c:
                    dv.append(f"{lab}/wave {c[name] / c['SQ_WAVES']:.0f}")
        if "TCC_HIT_sum" in c and c["TCC_HIT_sum"] + c.get("TCC_MISS_sum", 0):
            dv.append(f"L2 hit {c['TCC_HIT_sum'] / (c['TCC_HIT_sum'] + c['TCC_MISS_sum']):.3f}")
        if c.get("TCP_TCC_READ_REQ_sum") and "TCP_TCC_READ_REQ_LATENCY_sum" in c:
            dv.append(f"L1->L2 read latency {c['TCP_TCC_READ_REQ_LATENCY_sum'] / c['TCP_TCC_READ_REQ_sum']:.0f} cycles")
        if c.get("SQ_INSTS_VALU_MFMA_MOPS_F16"):  # counts F16 MFMA work in units of 512 FLOP
            dv.append(f"F16 MFMA {c['SQ_INSTS_VALU_MFMA_MOPS_F16'] * 512 / 1e12:.3f} TFLOP")
        if dv:
            out.append("  -> " + ", ".join(dv))
    return "\n".join(out)


def summarize_overlap(trace):
    """How much the kernels of different HIP streams overlap in a kernel
    trace: the time during which at least one kernel runs, the part of it
    with kernels of two or more streams in flight, and the time-weighted mean
    number of streams with a kernel in flight."""
    ev = []
    streams = set()
    for r in _csv_rows(trace, "kernel_trace.csv"):
        t0, t1, sid = int(r["Start_Timestamp"]), int(r["End_Timestamp"]), r["Stream_Id"]
        if t1 > t0:
            ev += [(t0, 1, sid), (t1, -1, sid)]
            streams.add(sid)
    ev.sort(key=lambda e: (e[0], e[1]))
    live = {}
    busy = multi = weighted = 0
    prev = None
    for t, d, sid in ev:
        if prev is not None:
            n = len(live)
            dt = t - prev
            if n >= 1:
                busy += dt
                weighted += n * dt
            if n >= 2:
                multi += dt
        live[sid] = live.get(sid, 0) + d
        if live[sid] == 0:
            del live[sid]
        prev = t
    return (f"streams with kernels: {len(streams)}\n"
            f"GPU busy (some kernel in flight): {busy / 1e6:.1f} ms\n"
            f"two or more streams in flight: {multi / 1e6:.1f} ms ({multi / max(busy, 1):.3f} of busy time)\n"
            f"mean streams in flight while busy: {weighted / max(busy, 1):.2f}")


def _profile_tag(tag):
    try:
        for ln in open(PROFILE_SUMMARY):
            if ln.startswith(tag):
                return float(ln[len(tag):])
    except OSError:
        pass
    return None


def traffic_per_ray():
    """The closest-hit kernel's measured bytes per ray from the committed
    counter summary (None when absent)."""
    return _profile_tag(TRAFFIC_TAG)


VALU_TAG = "VALU k_extend busy="


def copy_probe(mib):
    import torch

    n = mib * (1 << 20) // 4
    src = torch.ones(n, dtype=torch.float32, device="cuda:0")
    dst = torch.empty_like(src)
    torch.cuda.synchronize()
    for _ in range(5):
        dst.copy_(src)
    torch.cuda.synchronize()
    print(json.dumps({"copy_probe_bytes": n * 4, "launches": 5}), flush=True)


def make_scene(cfg, args):
    from radiantiumplusplus_amd import scenes

    if cfg == "large_mesh":
        b = scenes.large_mesh(grid=args.grid)
        name = f"large_mesh_terrain{args.grid}_256spheres_1080p_64spp"
    elif cfg == "many_balls":
        b = scenes.many_balls()
        name = "many_balls_64spheres_512x512_16spp"
    else:
        b = scenes.volume_box()
        name = "volume_box_perlin256_1024x1024_64spp"
    if args.spp:
        b.sampler["sample_count"] = args.spp
    return b, name


TILE = 16


def _tile_pixels(W, H, step):
    """Pixels in tiles 0, step, 2*step, ... of the row-major 16x16 tile list."""
    tx, ty = (W + TILE - 1) // TILE, (H + TILE - 1) // TILE
    n = 0
    for t in range(0, tx * ty, step):
        bx, by = (t % tx) * TILE, (t // tx) * TILE
        n += (min(bx + TILE, W) - bx) * (min(by + TILE, H) - by)
    return n


def _coprime_step(target, tiles_x):
    s = max(1, int(round(target)))
    while np.gcd(s, tiles_x) != 1:
        s += 1
    return s


def cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def cpu_baseline(b, seconds):
    """Time the oracle, all host threads, on an even subsample of the frame's
    16x16 tiles at full spp.  The tile stride is coprime to the tiles per
    row, so the subsample covers every row and column band of the image; it
    is calibrated so that the measured run takes about `seconds`.  Returns
    the baseline record and the rendered tiles (mean and sum of squares)."""
    sys.path.insert(0, os.path.join(ROOT, "tests"))
    import _oracle as O

    threads = len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else (os.cpu_count() or 1)
    t0 = time.time()
    o = O.OracleScene(b)
    build_s = time.time() - t0
    W, H = b.camera["width"], b.camera["height"]
    spp = b.sampler["sample_count"]
    tiles_x = (W + TILE - 1) // TILE
    ntiles = tiles_x * ((H + TILE - 1) // TILE)
    # calibration: enough tiles to keep every thread busy
    step = _coprime_step(max(1, ntiles // (8 * threads)), tiles_x)
    for _ in range(4):
        fb, sq, t = o.render(threads=threads, want_sumsq=True, tile_step=step)
        if t >= 0.5 * seconds or step == 1:
            break
        step = _coprime_step(max(1.0, step * t / seconds), tiles_x)
    samples = _tile_pixels(W, H, step) * spp
    rec = {
        "value": samples / t,
        "unit": "samples/s",
        "cores": threads,
        "kind": "port",
        "label": "vs refcpu (Embree unavailable)",
        "cpu_model": cpu_model(),
        "nproc": os.cpu_count(),
        "threads": threads,
        "accel": "binned-SAH BVH collapsed to 4-wide nodes, SSE slab tests, x86-64-v3 build (AVX2/FMA)"
                 if os.path.basename(O.LIB_PATH) == "librefcpu.so" else "4-wide SSE BVH, x86-64-v2 build",
        "sample": f"oracle {b.renderer['type']} integrator, 1 in {step} of the {ntiles} 16x16 tiles of the "
                  f"{W}x{H} frame at {spp} spp ({samples} samples, {t:.1f} s; BVH build {build_s:.1f} s excluded)",
    }
    return rec, fb, sq, step


def image_match(g_fb, g_sq, o_fb, o_sq, spp, step):
    """Per-tile z-test of the GPU frame against the oracle's tiles (the same
    16x16 tiles the CPU baseline rendered, both at the frame's spp) and the
    relMSE of their tile means."""
    H, W = g_fb.shape[:2]
    tiles_x = (W + TILE - 1) // TILE
    ntiles = tiles_x * ((H + TILE - 1) // TILE)
    zs, rels = [], []
    for t in range(0, ntiles, step):
        x0, y0 = (t % tiles_x) * TILE, (t // tiles_x) * TILE
        sl = (slice(y0, min(y0 + TILE, H)), slice(x0, min(x0 + TILE, W)))
        stats = []
        for fb, sq in ((g_fb, g_sq), (o_fb, o_sq)):
            m = fb[sl].astype(np.float64)
            var = np.maximum(sq[sl].astype(np.float64) / spp - m ** 2, 0.0) / spp
            stats.append((m.mean(axis=(0, 1)), var.sum(axis=(0, 1)) / m.shape[0] ** 2 / m.shape[1] ** 2))
        (ma, va), (mb, vb) = stats
        floor = (max(2e-6, 2 * spp * 2.0 ** -24) * np.maximum(np.abs(ma), np.abs(mb))) ** 2
        zs.append(np.abs(ma - mb) / np.sqrt(va + vb + floor + 1e-20))
        rels.append((ma - mb) ** 2 / (mb ** 2 + 1e-4))
    z, rel = np.array(zs), np.array(rels)
    return {"tiles": len(zs), "tile": f"{TILE}x{TILE}", "max_z": float(z.max()), "frac_z_over_4": float((z > 4).mean()),
            "relmse": float(rel.mean()), "spp_each": spp,
            "note": "GPU frame (another seed) vs the oracle's tiles of the CPU-baseline run, both at the frame's spp"}


def rel_mse(x, ref):
    return float(np.mean((x.astype(np.float64) - ref) ** 2 / (ref.astype(np.float64) ** 2 + 1e-2)))


def guiding_measure(ctx, scale=1.0, budget=256, ref_spp=4096, quirks=False):
    """Door-gap room, 1280x720: wall time for learned guiding (online
    training inside each render's own budget, from a fresh network) to reach
    the relMSE of the plain GPU tracer at `budget` spp, against a plain
    render at `ref_spp`.  Guided renders are timed at budgets on a grid of
    8 spp (binary search for the smallest whose relMSE is at most plain's);
    both errors are taken against the same reference, so its own noise
    enters both alike.  With the reference's quirks on, visible-normal GGX
    vertices (the glossy boxes) are not guided: their sample density is not
    their pdf."""
    from radiantiumplusplus_amd import _ffi as F
    from radiantiumplusplus_amd import hip, scenes

    W, H = int(1280 * scale), int(720 * scale)
    b = scenes.guiding_room(width=W, height=H, spp=budget)
    s = hip.Scene.from_builder(ctx, b)
    fl = 0 if quirks else F.RAD_RENDER_FIX_QUIRKS
    ref, _, _ = s.render(b.render_desc(spp=ref_spp, seed=7, flags=fl))
    s.render(b.render_desc(spp=16, seed=3, flags=fl))  # first-use costs out of the timings
    t = time.time()
    plain, _, _ = s.render(b.render_desc(spp=budget, seed=8, flags=fl))
    t_plain = time.time() - t
    e_p = rel_mse(plain, ref)

    def guided(spp):
        s.set_guide_params(None)
        d = b.render_desc(spp=spp, seed=9, flags=fl)
        d.guiding = 1
        t0 = time.time()
        img, _, st = s.render(d)
        return time.time() - t0, rel_mse(img, ref), st

    runs = {}

    def run(k):  # k units of 8 spp
        r = guided(8 * k)
        runs[8 * k] = r
        return r

    kb = budget // 8
    best = run(kb)
    e_g_budget = best[1]
    lo, hi, reached = 0, kb, best[1] <= e_p
    while not reached and hi < 4 * kb:  # guided worse than plain at equal spp: raise its budget
        lo, hi = hi, 2 * hi
        best = run(hi)
        reached = best[1] <= e_p
    while reached and hi - lo > 1:  # smallest budget on the grid that reaches plain's error
        mid = (lo + hi) // 2
        r = run(mid)
        if r[1] <= e_p:
            hi, best = mid, r
        else:
            lo = mid
    t_eq, e_eq, st_eq = best
    spp_eq = 8 * hi
    return {
        "workload": f"guiding_room_{W}x{H}_quirks_{'on' if quirks else 'off'}",
        "plain_spp": budget,
        "plain_relmse": e_p,
        "plain_s": t_plain,
        "guided_relmse_at_plain_spp": e_g_budget,
        "relmse_ratio_equal_spp": e_g_budget / e_p,
        "guided_spp_to_plain_relmse": spp_eq if reached else None,
        "guided_relmse_there": e_eq,
        "guided_s_to_plain_relmse": t_eq if reached else None,
        "time_ratio_guided_over_plain": (t_eq / t_plain) if reached else None,
        "method": "timed guided renders from a fresh network on an 8-spp grid (binary search), smallest budget "
                  "whose relMSE is at most the plain render's; no extrapolation",
        "trials": {str(k): [round(v[0], 3), v[1]] for k, v in sorted(runs.items())},  # spp: [s, relMSE]
        "reference": f"plain GPU render at {ref_spp} spp (the room's plain GPU render is tested against the oracle)",
        "guide_steps": st_eq.guide_steps,
        "guide_records": st_eq.guide_records,
        "guide_final_loss": st_eq.guide_loss,
    }


def serving_measure(ctx, n_requests=40, rate=20.0):
    """Seeded Poisson stream (mean 20 req/s) over resident scenes of the
    many-balls, large-mesh and volume workloads; resolution, spp and guiding
    drawn per request."""
    from radiantiumplusplus_amd import hip, scenes, serve

    builders = {"many_balls": scenes.many_balls(), "large_mesh": scenes.large_mesh(),
                "volume_box": scenes.volume_box()}
    res = {k: hip.Scene.from_builder(ctx, b) for k, b in builders.items()}
    specs = serve.poisson_requests(n_requests, rate=rate, seed=4)
    srv = serve.Server(ctx, hbm_budget=64 << 30, max_inflight=8)
    out = serve.run_stream(srv, res, builders, specs)
    st = srv.stats()
    srv.close()
    lat = np.array([r.times.latency_ms for r in out])
    return {
        "workload": f"poisson_{rate:g}rps_{n_requests}req_seed4",
        "requests": n_requests,
        "completed": int(st.completed),
        "samples_per_s": st.samples_per_s,
        "p50_ms": st.p50_ms,
        "p99_ms": st.p99_ms,
        "mean_ms": st.mean_ms,
        "max_ms": float(lat.max()),
        "peak_hbm_bytes": int(st.peak_held_bytes),
    }


def main():
    args = parse()
    if args.gpus != 1:
        print(json.dumps({"error": "this benchmark runs on one GPU; --gpus above 1 is not supported (sample-space sharding is a design only)",
                          "n_gpus": args.gpus}))
        sys.exit(2)
    if args.copy_probe:
        return copy_probe(args.copy_probe)
    if args.summarize:
        print(summarize(args.summarize))
        return
    if args.summarize_counters:
        print(summarize_counters(args.summarize_counters))
        return
    if args.summarize_overlap:
        print(summarize_overlap(args.summarize_overlap))
        return
    if args.serving_only:
        from radiantiumplusplus_amd import hip

        print(json.dumps(serving_measure(hip.Context(0))), flush=True)
        return
    if args.guiding_only:
        from radiantiumplusplus_amd import hip

        print(json.dumps(guiding_measure(hip.Context(0), args.guide_scale)), flush=True)
        return
    from radiantiumplusplus_amd import _ffi as F
    from radiantiumplusplus_amd import hip

    t0 = t0_all = time.time()
    b, name = make_scene(args.config, args)
    gen_s = time.time() - t0
    ctx = hip.Context(0)
    t0 = time.time()
    scene = hip.Scene.from_builder(ctx, b, builder=F.RAD_BVH_DEVICE if args.builder == "device" else F.RAD_BVH_HOST)
    setup_s = time.time() - t0
    info = scene.info()
    W, H = b.camera["width"], b.camera["height"]
    spp = b.sampler["sample_count"]
    tune = None
    launch = [int(x) for x in args.launch.split(",")] if args.launch else None
    if launch is None and not args.no_autotune:
        # launch configuration picked by timing short renders (images do not depend on it)
        rep = scene.autotune(b.render_desc(spp=max(1, min(spp, (128 << 20) // (W * H))), seed=1))
        tune = {"path_slots": rep.path_slots, "blocks_per_cu": rep.blocks_per_cu,
                "trace_blocks_per_cu": rep.trace_blocks_per_cu,
                "trials": [[t.path_slots, t.blocks_per_cu, t.trace_blocks_per_cu, round(t.ms, 3)]
                           for t in rep.trial[:rep.trials]]}
        print(f"# autotune: slots {rep.path_slots}, blocks/CU {rep.blocks_per_cu}, "
              f"trace blocks/CU {rep.trace_blocks_per_cu}", file=sys.stderr, flush=True)
    rd = b.render_desc(spp=spp, seed=1, flags=F.RAD_RENDER_PROFILE | (F.RAD_RENDER_UNSORTED if args.unsorted else 0))
    if launch:
        rd.path_slots, rd.blocks_per_cu, rd.trace_blocks_per_cu = launch
    print(f"# scene {name}: {info.primitive_count} primitives, {info.node_count} BVH nodes, "
          f"build {info.bvh_build_ms:.0f} ms, generation {gen_s:.1f} s, upload+build {setup_s:.1f} s",
          file=sys.stderr, flush=True)
    for i in range(args.warmup):
        _, _, st = scene.render(rd)
        print(f"# warmup {i}: {st.render_ms:.1f} ms (t = {time.time() - t0_all:.1f} s)", file=sys.stderr, flush=True)
    times, stats = [], []
    t_all = time.time()
    for i in range(args.steps):
        rd.seed = 100 + i
        t = time.time()
        _, _, st = scene.render(rd)
        times.append(time.time() - t)
        stats.append(st)
        print(f"# step {i}: {times[-1] * 1e3:.1f} ms (render {st.render_ms:.1f} ms), {st.segments} segments, "
              f"{st.iterations} iterations", file=sys.stderr, flush=True)
    total = time.time() - t_all
    samples = W * H * spp * args.steps
    ms_step = 1e3 * total / args.steps
    ext_ms = sum(s.kernel_ms[F.RAD_KERNEL_EXTEND] for s in stats)
    ext_launch = sum(s.kernel_launches[F.RAD_KERNEL_EXTEND] for s in stats)
    segs = sum(s.segments for s in stats)
    achieved = TRACE_BYTES_PER_RAY * segs / (ext_ms * 1e-3) / 1e9 if ext_ms > 0 else 0.0
    out = {
        "metric": METRIC,
        "value": samples / total,
        "unit": "samples/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": ms_step,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "value_note": "value = samples/s of the plain GPU path on the workload below; the guided-vs-plain "
                      "time to equal relMSE is under guiding, p50/p99 request latency under serving",
        "dtype": "f32",
        "data": "synthetic",
        "config": {
            "workload": name,
            "width": W,
            "height": H,
            "spp": spp,
            "max_depth": b.renderer["max_depth"],
            "primitives": int(info.primitive_count),
            "integrator": b.renderer["type"],
        },
        "roofline": {
            "bound": "hbm",
            "kernel": "k_extend (closest-hit traversal)",
            "achieved": achieved,
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": achieved / HBM_PEAK_GBS,
            "traffic": (traffic_per_ray() * segs / max(ext_launch, 1)) if traffic_per_ray() else None,
            "traffic_note": "bytes per launch beyond L2: FETCH_SIZE + WRITE_SIZE per traced ray from the rocprofv3 "
                            "--pmc runs in profiles/k_extend_large_mesh.txt (scaled by a plain copy), times this "
                            "run's rays per launch",
            "avg_launch_ms": ext_ms / max(ext_launch, 1),
            "valu_busy": _profile_tag(VALU_TAG),
            "valu_note": "fraction of SIMD cycles issuing VALU instructions in k_extend (SQ_ACTIVE_INST_VALU, "
                         "GRBM_GUI_ACTIVE in profiles/k_extend_large_mesh.txt): the kernel is bound by instruction "
                         "issue and the latency of its node reads, not by HBM bandwidth",
            "launch": {"path_slots": stats[0].slots, "blocks_per_cu": stats[0].blocks_per_cu,
                       "trace_blocks_per_cu": stats[0].trace_blocks_per_cu},
            "rays_per_s": segs / (ext_ms * 1e-3) if ext_ms > 0 else 0.0,
        },
        "stats": {
            "segments_per_step": segs / args.steps,
            "shadow_rays_per_step": sum(s.shadow_rays for s in stats) / args.steps,
            "iterations_per_step": sum(s.iterations for s in stats) / args.steps,
            "slots": stats[0].slots,
            "kernel_ms_per_step": {k: sum(s.kernel_ms[i] for s in stats) / args.steps
                                   for i, k in enumerate(["regen", "extend", "shade", "shadow", "guide", "train"])},
            "bvh_build_ms": info.bvh_build_ms,
            "bvh_depth": int(info.bvh_depth),
            "bvh_stack_need": int(info.bvh_stack_need),
            "bvh_builder": args.builder,
            "material_sorted": not args.unsorted,
            "autotune": tune,
        },
    }
    if args.config == "large_mesh" and not args.no_guiding:
        print("# guided vs plain (door-gap room)", file=sys.stderr, flush=True)
        out["guiding"] = guiding_measure(ctx, args.guide_scale)
        out["guiding_quirks_on"] = guiding_measure(ctx, args.guide_scale, quirks=True)
    if args.config == "large_mesh" and not args.no_serving:
        print("# serving stream", file=sys.stderr, flush=True)
        out["serving"] = serving_measure(ctx, args.serve_requests)
    if not args.no_cpu:
        cb, ofb, osq, step = cpu_baseline(b, args.cpu_seconds)
        out["cpu_baseline"] = cb
        out["gpu_over_cpu"] = out["value"] / cb["value"]
        out["gpu_over_cpu_label"] = "vs refcpu (Embree unavailable)"
        rd_m = b.render_desc(spp=spp, seed=999, flags=F.RAD_RENDER_WANT_SUMSQ)
        gfb, gsq, _ = scene.render(rd_m, want_sumsq=True)
        out["image_match"] = image_match(gfb, gsq, ofb, osq, spp, step)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
