"""Benchmark: SU(3) link updates/s and % of HBM roofline at 32^4.

Workload (one "step"): one iteration of quenched SU(3) ensemble generation on a
32^4 lattice at beta=6.0 from a cold start, FP32 links in 12-real storage --
1 heatbath sweep + 4 overrelaxation sweeps (8 (parity, mu) launches each),
reunitarisation, plaquette and Polyakov loop with FP64 accumulation -- captured in
a hipGraph and replayed.  value = link updates per second of the whole job
(5 * 4V updates per step).  Inputs are resident in HBM before timing starts.

Prints ONE JSON line.  Extra objects:
  roofline      dominant kernel (the overrelaxation launch): algorithmic bytes
                9 * 48 B per link update x V/2 updates per launch, divided by the
                launch's average duration measured with HIP events on its stream
  cpu_baseline  the FP64 oracle on this host's cores, one iteration at 32^4
  plain_fp64    the plain single-lattice path (FP64 18-real, eager launches)
  precision     FP32-12 vs FP64-18: lockstep per-iteration plaquette / Polyakov
                differences and free-chain ensemble means
  operator_loops  operator-basis Wilson loops (A0 measurement at 32^4 FP64, 33
                family at r = 12) with the correlator launch's roofline
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_HBM_GBS = 8000.0
PEAK_F64_TFS = 78.6  # FP64 matrix
DIMS = (32, 32, 32, 32)
BETA = 6.0


def profile_traffic(shape):
    """HBM bytes per overrelaxation launch measured by rocprofv3 FETCH_SIZE/WRITE_SIZE
    passes (calibrated against a device copy) for this launch shape, from the summary
    committed under profiles/; None when no summary matches the shape."""
    key = (f"kernel=overrelaxation block={shape['block']} brick={','.join(map(str, shape['brick']))} "
           f"lds={shape['lds']} piped={shape['piped']} bytes=")
    pdir = os.path.join(ROOT, "profiles")
    if not os.path.isdir(pdir):
        return None, None
    for name in sorted(os.listdir(pdir)):
        if not name.endswith(".md"):
            continue
        for line in open(os.path.join(pdir, name)):
            if line.startswith("traffic-per-launch: ") and key in line:
                return int(line.split("bytes=")[1].split()[0]), f"profiles/{name}"
    return None, None


PROFILE_32 = "su3_32x4_f32_12_iteration_kernels.md"
PROFILE_64 = "su3_64x4_f32_8_iteration_kernels.md"


def profiled_shapes(name):
    """The overrelaxation and heatbath launch shapes the committed rocprof summary
    profiles/<name> was taken with, or None.  The benchmark runs its lattices with
    them, so the summary's traffic is that of the launches timed here (left to the
    autotuner, near-equal shapes can differ from one run to the next)."""
    path = os.path.join(ROOT, "profiles", name)
    if not os.path.exists(path):
        return None
    for line in open(path):
        if line.startswith("Tuned shapes: overrelaxation "):
            body = line[len("Tuned shapes: overrelaxation "):].rstrip().rstrip(".")
            or_part, hb_part = body.split(", heatbath ")
            return {"overrelax": json.loads(or_part), "heatbath": json.loads(hb_part), "source": f"profiles/{name}"}
    return None


def pin_shapes(lat, shapes):
    """set the lattice's launch shapes (marks it tuned); returns their source"""
    if not shapes:
        return "autotuner"
    for kernel, key in ((1, "overrelax"), (0, "heatbath")):
        c = shapes[key]
        lat.set_launch(kernel, c["block"], tuple(c["brick"]), c["lds"], c["piped"])
    return shapes["source"]


def link_bytes(nc, storage, prec):
    return (2 * nc * nc if storage == 18 else storage) * prec


def time_launches(sun_amd, lat, stream, hb: bool, reps: int) -> float:
    """average duration (ms) of one (parity, mu) update launch, HIP events on its stream"""
    t = sun_amd.Timer()
    for _ in range(2):  # warm
        if hb:
            lat.heatbath_sub(1, 0, 0, 0, stream)
        else:
            lat.overrelax_sub(0, 0, stream)
    t.start(stream)
    for r in range(reps):
        parity, mu = (r // 4) % 2, r % 4
        if hb:
            lat.heatbath_sub(1, r, parity, mu, stream)
        else:
            lat.overrelax_sub(parity, mu, stream)
    t.stop(stream)
    ms = t.ms() / reps
    t.close()
    return ms


def cpu_baseline(min_seconds: float = 10.0, max_iters: int = 20):
    """FP64 oracle on this host's cores: whole iterations (1 HB + 4 OR sweeps) of the
    same 32^4 workload until at least min_seconds have passed."""
    from oracle import oracle as o
    cores = min(os.cpu_count() or 1, 16)
    o.set_threads(cores)
    U = o.cold_start(3, DIMS)
    # one heatbath sweep first so the timed iterations start from a non-trivial field
    o.heatbath_sweep(U, DIMS, BETA, 2, 0)
    n = 0
    t0 = time.perf_counter()
    while n < max_iters and (n == 0 or time.perf_counter() - t0 < min_seconds):
        o.heatbath_sweep(U, DIMS, BETA, 2, 1 + n)
        for _ in range(4):
            o.overrelax_sweep(U, DIMS)
        n += 1
    dt = time.perf_counter() - t0
    V = int(np.prod(DIMS))
    # one thread, on a 16^4 lattice (the same per-site work; a 32^4 iteration would
    # take ~20 s on one core)
    o.set_threads(1)
    small = (16, 16, 16, 16)
    W = o.cold_start(3, small)
    o.heatbath_sweep(W, small, BETA, 2, 0)
    n1 = 0
    t1 = time.perf_counter()
    while n1 < 10 and (n1 == 0 or time.perf_counter() - t1 < 3.0):
        o.heatbath_sweep(W, small, BETA, 2, 1 + n1)
        for _ in range(4):
            o.overrelax_sweep(W, small)
        n1 += 1
    dt1 = time.perf_counter() - t1
    o.set_threads(cores)
    model = ""
    try:
        with open("/proc/cpuinfo") as f:
            model = next((ln.split(":", 1)[1].strip() for ln in f if ln.startswith("model name")), "")
    except OSError:
        pass
    return {"value": n * 5 * 4 * V / dt, "unit": "link-updates/s", "cores": cores, "kind": "port",
            "sample": f"FP64 oracle (C, OpenMP, {cores} threads): {n} iterations of 1 heatbath + 4 "
                      f"overrelaxation sweeps of SU(3) 32^4 beta=6.0 (after one heatbath sweep from cold), "
                      f"{dt:.1f} s",
            "single_thread": {"value": n1 * 5 * 4 * int(np.prod(small)) / dt1, "unit": "link-updates/s",
                              "sample": f"{n1} iterations of SU(3) 16^4 on one thread, {dt1:.1f} s"},
            "host": {"cpu_model": model, "nproc": os.cpu_count()}}


def batch_means(x, nblocks=10):
    """mean and its standard error from nblocks block means (autocorrelated chain)"""
    x = np.asarray(x, dtype=np.float64)
    n = len(x) // nblocks * nblocks
    b = x[len(x) - n:].reshape(nblocks, -1).mean(axis=1)
    return float(b.mean()), float(b.std(ddof=1) / np.sqrt(nblocks))


def plain_fp64_leg(sun_amd, ctx, stream, value, updates_per_step, n=25):
    """The plain single-lattice path -- FP64 18-real, one kernel per (parity, mu),
    eager launches, reunitarize + plaquette + Polyakov every iteration -- on the same
    chain (seed, sweeps, cold start) as the FP32 run.  Its first iteration (where the
    autotuner times its launch shapes) runs before the clock starts."""
    with sun_amd.Lattice(ctx, 3, DIMS, BETA, 18, 8) as pl:
        pl.cold_start(stream)
        pl.generate(seed=2, n_iter=1, n_or=4, reunit_every=1, use_graph=False, stream=stream)
        sun_amd.sync(stream)
        t0 = time.perf_counter()
        pl.generate(seed=2, n_iter=n, n_or=4, reunit_every=1, first_sweep=1, use_graph=False, stream=stream)
        sun_amd.sync(stream)
        pv = updates_per_step * n / (time.perf_counter() - t0)
    return {"value": pv, "unit": "link-updates/s", "iterations": n,
            "config": "SU(3) 32^4 beta=6.0 cold start, FP64 18-real, one kernel per (parity, mu), eager "
                      "launches, reunitarize + plaquette + Polyakov every iteration; tuned before timing",
            "gain": value / pv}


def precision_leg(sun_amd, ctx, stream, shapes, n_lock=200):
    """FP32 12-real against FP64 18-real at 32^4 (beta 6.0, cold start, seed 2).
    Lockstep: every iteration of the FP64 chain is also run in FP32 from the same
    field (the FP64 field converted on the device to FP32 12-real), and the two
    iterations' plaquettes and Polyakov loops are compared -- the error of one FP32
    iteration, which free-running chains cannot show (a sweep amplifies differences
    ~100x, so they separate after a few iterations).  Ensemble: the FP32 chain run
    free beside the FP64 chain, means over the second half with batch-means errors."""
    V = int(np.prod(DIMS))
    dp, dl, p64, l64 = [], [], [], []
    with sun_amd.Lattice(ctx, 3, DIMS, BETA, 18, 8) as l64_lat, sun_amd.Lattice(ctx, 3, DIMS, BETA, 12, 4) as l32:
        pin_shapes(l32, shapes)
        l64_lat.cold_start(stream)
        for it in range(n_lock):
            l32.convert_from(l64_lat, stream)
            o32 = l32.generate(seed=2, n_iter=1, n_or=4, reunit_every=1, first_sweep=it, use_graph=False,
                               stream=stream)
            o64 = l64_lat.generate(seed=2, n_iter=1, n_or=4, reunit_every=1, first_sweep=it, use_graph=False,
                                   stream=stream)
            dp.append(float(np.abs(o32[0, :2] - o64[0, :2]).max()))
            dl.append(abs(complex(o32[0, 2], o32[0, 3]) - complex(o64[0, 2], o64[0, 3])))
            p64.append(float(o64[0, :2].mean()))
            l64.append(abs(complex(o64[0, 2], o64[0, 3])))
        l32.cold_start(stream)
        free = l32.generate(seed=2, n_iter=n_lock, n_or=4, reunit_every=1, first_sweep=0, stream=stream)
    dp, dl = np.array(dp), np.array(dl)
    half = n_lock // 2
    p32 = free[:, :2].mean(axis=1)
    m32, e32 = batch_means(p32[half:])
    m64, e64 = batch_means(np.array(p64)[half:])
    a32, ae32 = batch_means(np.hypot(free[half:, 2], free[half:, 3]))
    a64, ae64 = batch_means(np.array(l64)[half:])
    return {"lockstep": {"iterations": n_lock,
                         "plaquette_absdiff_max": float(dp.max()), "plaquette_absdiff_mean": float(dp.mean()),
                         "plaquette_absdiff_median": float(np.median(dp)),
                         "iterations_over_1e-6": int((dp > 1e-6).sum()),
                         "fraction_within_1e-6": float((dp <= 1e-6).mean()),
                         "polyakov_absdiff_max": float(dl.max()), "polyakov_absdiff_mean": float(dl.mean()),
                         "target": 1e-6,
                         "note": "each FP32-12 iteration (HB + 4 OR + reunit + plaquette + Polyakov) starts from "
                                 "the FP64-18 chain's field of the same iteration; plaquette difference = max over "
                                 "the spatial and temporal components.  Iterations whose heatbath flips an "
                                 "accept/reject decision against FP64 (the FP32 staple moves a near-tie; ~1 in 5 "
                                 "iterations at 32^4) carry the O(1) change of that link and its cascade through "
                                 "the sweep into the plaquette"},
            "ensemble": {"window": [half, n_lock],
                         "plaquette_mean_f32": [m32, e32], "plaquette_mean_f64": [m64, e64],
                         "plaquette_mean_diff": m32 - m64, "plaquette_mean_diff_sigma": float(np.hypot(e32, e64)),
                         "abs_polyakov_mean_f32": [a32, ae32], "abs_polyakov_mean_f64": [a64, ae64],
                         "abs_polyakov_mean_diff": a32 - a64, "abs_polyakov_mean_diff_sigma": float(np.hypot(ae32, ae64)),
                         "note": "FP32-12 chain run free beside the FP64-18 chain (same seed and sweeps); "
                                 "batch-means errors over 10 blocks"},
            "lattice": list(DIMS), "beta": BETA, "volume": V}


def large_leg(sun_amd, ctx, stream, n_iter=6, warm=2, shapes=None):
    """SU(3) 64^4 (16.7M sites, 2.15 GB of links), beta=6.2, FP32 8-real links from a
    Haar start (8 reals cannot hold a cold start); iterations of 1 heatbath + 4
    overrelaxation sweeps + plaquette + Polyakov loop (FP64 sums), graph replay.
    Reports link updates/s and the overrelaxation launch's algorithmic GB/s
    (9 x 32 B per update) from HIP events."""
    dims = (64, 64, 64, 64)
    V = int(np.prod(dims))
    with sun_amd.Lattice(ctx, 3, dims, 6.2, 8, 4) as lat:
        shape_source = pin_shapes(lat, shapes)
        lat.hot_start(3, stream)
        lat.generate(seed=3, n_iter=warm, n_or=4, reunit_every=0, stream=stream)
        sun_amd.sync(stream)
        t0 = time.perf_counter()
        obs = lat.generate(seed=3, n_iter=n_iter, n_or=4, reunit_every=0, first_sweep=warm, stream=stream)
        sun_amd.sync(stream)
        dt = time.perf_counter() - t0
        or_ms = time_launches(sun_amd, lat, stream, hb=False, reps=16)
        hb_ms = time_launches(sun_amd, lat, stream, hb=True, reps=8)
        per_launch = 9 * 32 * (V // 2)
        return {"value": 5 * 4 * V * n_iter / dt, "unit": "link-updates/s", "iterations": n_iter,
                "ms_per_iteration": dt / n_iter * 1e3,
                "overrelax_launch_ms": or_ms, "overrelax_gbs": per_launch / (or_ms * 1e-3) / 1e9,
                "overrelax_frac": per_launch / (or_ms * 1e-3) / 1e9 / PEAK_HBM_GBS,
                "heatbath_launch_ms": hb_ms, "heatbath_gbs": per_launch / (hb_ms * 1e-3) / 1e9,
                "launch_shape": lat.get_launch(1).as_dict(), "heatbath_launch_shape": lat.get_launch(0).as_dict(),
                "launch_shape_source": shape_source,
                "plaquette_last": [float(obs[-1, 0]), float(obs[-1, 1])],
                "polyakov_last": [float(obs[-1, 2]), float(obs[-1, 3])],
                "config": "SU(3) 64^4 beta=6.2 Haar start, FP32 8-real links; iteration = HB + 4 OR + "
                          "plaquette + spatially averaged Polyakov loop (FP64 sums), hipGraph replay"}


XGMI_LINK_GBS = 153.0  # one xGMI link of an MI355X, per direction


def shard_leg(sun_amd, ctx, stream, n_iter=4, warm=2):
    """One GPU's share of the 64^4 FP32-8 lattice split 8 ways: 64 x 64 x 8 x 64 (split
    in x2, spatial, so Polyakov lines stay on one GPU) and 64^3 x 8 (split in t), run
    periodic as a stand-in for the share.  A split lattice would exchange, after every
    (parity, mu) launch, one plane of the just-updated U_mu links with each of its two
    neighbours; the leg reports the local launch time beside that face's bytes and its
    time on one xGMI link, i.e. how much interior work there is to hide the exchange."""
    out = {}
    for name, dims, d in (("x2_split_64x64x8x64", (64, 64, 8, 64), 2), ("t_split_64x64x64x8", (64, 64, 64, 8), 3)):
        V = int(np.prod(dims))
        with sun_amd.Lattice(ctx, 3, dims, 6.2, 8, 4) as lat:
            lat.hot_start(3, stream)
            lat.generate(seed=3, n_iter=warm, n_or=4, reunit_every=0, stream=stream)
            sun_amd.sync(stream)
            t0 = time.perf_counter()
            lat.generate(seed=3, n_iter=n_iter, n_or=4, reunit_every=0, first_sweep=warm, stream=stream)
            sun_amd.sync(stream)
            dt = time.perf_counter() - t0
            or_ms = time_launches(sun_amd, lat, stream, hb=False, reps=16)
        face = V // dims[d] // 2 * 32  # one plane of U_mu at one parity, 8-real FP32
        out[name] = {"lattice": list(dims), "ms_per_iteration": dt / n_iter * 1e3,
                     "overrelax_launch_ms": or_ms, "face_bytes_per_launch": face,
                     "xgmi_ms_per_face": face / (XGMI_LINK_GBS * 1e9) * 1e3,
                     "exchange_to_launch": face / (XGMI_LINK_GBS * 1e9) * 1e3 / or_ms}
    out["note"] = ("periodic local lattice as the share; the exchange (2 faces, one per neighbour link, "
                   "both directions) and its overlap with interior sites are not run on one GPU")
    return out


BATCH_VOLUMES = [(8, 8, 8, 8), (12, 12, 12, 12), (16, 16, 16, 16), (16, 16, 16, 32), (24, 24, 24, 24)]


def batched_leg(sun_amd, ctx, stream, n_lat=64, n_iter=30, warm=3):
    """64 independent SU(3) lattices, volumes drawn from BATCH_VOLUMES, beta uniform in
    [5.7, 6.3], hot/cold starts 50/50, FP32 12-real; hipGraph-captured iterations of
    1 heatbath + 4 overrelaxation sweeps (one launch per (parity, mu) for all 64) +
    reunitarize + per-lattice plaquette."""
    rng = np.random.default_rng(4)
    vols = [BATCH_VOLUMES[i] for i in rng.integers(0, len(BATCH_VOLUMES), n_lat)]
    betas = rng.uniform(5.7, 6.3, n_lat)
    hot = rng.integers(0, 2, n_lat)
    lats = [sun_amd.Lattice(ctx, 3, v, float(b), 12, 4) for v, b in zip(vols, betas)]
    for i, l in enumerate(lats):
        if hot[i]:
            l.hot_start(1000 + i, stream)
        else:
            l.cold_start(stream)
    batch = sun_amd.Batch(ctx, lats, [4000 + i for i in range(n_lat)])
    batch.generate(first_sweep=0, n_iter=warm, n_or=4, reunit_every=1, stream=stream)
    sun_amd.sync(stream)
    t0 = time.perf_counter()
    obs = batch.generate(first_sweep=warm, n_iter=n_iter, n_or=4, reunit_every=1, stream=stream)
    sun_amd.sync(stream)
    dt = time.perf_counter() - t0
    sites = sum(int(np.prod(v)) for v in vols)
    # one overrelaxation sweep of all 64 lattices (8 batched launches), HIP events on
    # its stream: algorithmic bytes 9 * 48 B per link update, 4 * sites updates
    t = sun_amd.Timer()
    batch.overrelax(stream)
    t.start(stream)
    reps = 10
    for _ in range(reps):
        batch.overrelax(stream)
    t.stop(stream)
    or_sweep_ms = t.ms() / reps
    t.close()
    or_gbs = 9 * link_bytes(3, 12, 4) * 4 * sites / (or_sweep_ms * 1e-3) / 1e9
    # the single 32^4 FP32-12 lattice's overrelaxation launch (context launch shapes)
    # timed right after: the device runs a few % slower here, after the legs before
    # this one, than where the headline is measured
    with sun_amd.Lattice(ctx, 3, (32, 32, 32, 32), 6.0, 12, 4) as sl:
        sl.cold_start(stream)
        sl.generate(seed=2, n_iter=2, n_or=4, reunit_every=1, stream=stream)
        single_ms = time_launches(sun_amd, sl, stream, hb=False, reps=32)
    single_frac = 9 * link_bytes(3, 12, 4) * (32 ** 4 // 2) / (single_ms * 1e-3) / 1e9 / PEAK_HBM_GBS
    shapes = {k: dict(zip(("piped", "brick", "lds"), batch.get_launch(i)))
              for i, k in enumerate(("heatbath", "overrelax"))}
    batch.close()
    for l in lats:
        l.close()
    # algorithmic bytes of an iteration: HB + 4 OR (9 link transfers per update, 5 x 4
    # updates per site), reunitarisation (2 per link) and plaquette (1 per link)
    it_bytes = 4 * sites * link_bytes(3, 12, 4) * (45 + 2 + 1)
    return {"value": 5 * 4 * sites * n_iter / dt, "unit": "link-updates/s", "lattices": n_lat,
            "total_sites": sites, "iterations": n_iter, "ms_per_iteration": dt / n_iter * 1e3,
            "iteration_frac": it_bytes * n_iter / dt / 1e9 / PEAK_HBM_GBS,
            "overrelax_sweep_ms": or_sweep_ms, "overrelax_gbs": or_gbs, "overrelax_frac": or_gbs / PEAK_HBM_GBS,
            "single_32x4_overrelax_frac_same_point": single_frac,
            "launch_shapes": shapes,
            "plaquette_range_last": [float(obs[-1, :, :].mean(axis=1).min()),
                                     float(obs[-1, :, :].mean(axis=1).max())],
            "config": "64 SU(3) lattices, volumes from {8^4,12^4,16^4,16^3x32,24^4} (numpy seed 4), beta "
                      "U[5.7,6.3], hot/cold 50/50, FP32 12-real, hipGraph iteration = HB + 4 OR + reunit + "
                      "per-lattice plaquette"}


def batch_classes(sun_amd, ctx, stream, n_lat=64, reps=10, calibrate=False):
    """The 64-lattice batch of batched_leg broken down by volume class: one
    overrelaxation sweep (8 batched launches, the batch's default launch shapes) of
    the whole batch, then of each class's lattices as a batch of their own, timed with
    HIP events; algorithmic bytes 9 x 48 B per link update.  calibrate: two plain
    copies of the 201 MB 32^4 FP32-12 field first (the size reference for counter
    passes)."""
    rng = np.random.default_rng(4)
    vols = [BATCH_VOLUMES[i] for i in rng.integers(0, len(BATCH_VOLUMES), n_lat)]
    betas = rng.uniform(5.7, 6.3, n_lat)
    lats = [sun_amd.Lattice(ctx, 3, v, float(b), 12, 4) for v, b in zip(vols, betas)]
    for i, l in enumerate(lats):
        l.hot_start(1000 + i, stream)
    if calibrate:
        with sun_amd.Lattice(ctx, 3, DIMS, BETA, 12, 4) as a, sun_amd.Lattice(ctx, 3, DIMS, BETA, 12, 4) as b:
            for _ in range(2):
                b.copy_from(a, stream)
            sun_amd.sync(stream)

    def sweep(group):
        b = sun_amd.Batch(ctx, group, list(range(len(group))))
        b.overrelax(stream)
        sun_amd.sync(stream)
        t = sun_amd.Timer()
        t.start(stream)
        for _ in range(reps):
            b.overrelax(stream)
        t.stop(stream)
        ms = t.ms() / reps
        t.close()
        b.close()
        sites = sum(l.V for l in group)
        gbs = 9 * 48 * 4 * sites / (ms * 1e-3) / 1e9
        return {"lattices": len(group), "sites": sites, "overrelax_sweep_ms": ms, "gbs": gbs,
                "frac": gbs / PEAK_HBM_GBS}

    out = {"all": sweep(lats)}
    for v in sorted(set(vols)):
        out["x".join(map(str, v))] = sweep([l for l, vv in zip(lats, vols) if vv == v])
    for l in lats:
        l.close()
    return out


SERVE_VOLUMES = [(8, 8, 8, 8), (12, 12, 12, 12), (16, 16, 16, 16), (24, 24, 24, 24), (32, 32, 32, 32)]
SERVE_BETA = {2: (2.2, 2.6), 3: (5.6, 6.2), 4: (10.5, 11.2)}


def served_leg(sun_amd, ctx, n_jobs, util=0.75, budget=64 << 30):
    """Poisson arrivals of ensemble jobs (SU(2)/SU(3)/SU(4), volumes 8^4..32^4, beta in
    the usual range per N, 50..500 iterations of 1 HB + 4 OR + reunit + plaquette +
    Polyakov, FP32 links, FP64 reductions) into the job server's background loop.
    The arrival rate targets `util` of the device from each job's service time, modelled
    by a measured rate per (N, volume).  Latency = completion - submission."""
    rng = np.random.default_rng(5)
    jobs = []
    for j in range(n_jobs):
        nc = int(rng.integers(2, 5))
        dims = SERVE_VOLUMES[int(rng.integers(0, len(SERVE_VOLUMES)))]
        lo, hi = SERVE_BETA[nc]
        storage = 12 if nc == 3 else 18
        jobs.append(dict(nc=nc, dims=dims, beta=float(rng.uniform(lo, hi)), storage=storage, precision=4,
                         seed=5000 + j, hot_start=bool(rng.integers(0, 2)), n_iter=int(rng.integers(50, 501))))
    # service-time model measured on this device: one 20-iteration job of every (N,
    # volume) class run alone through a server; the arrival rate then targets `util`
    # of the device if the jobs ran one at a time (batching makes it less)
    calib = {}
    with sun_amd.Server(ctx, budget, max_jobs=16) as cs:
        cs.start()
        for nc in (2, 3, 4):
            for dims in SERVE_VOLUMES:
                jid = cs.submit(nc, dims, float(np.mean(SERVE_BETA[nc])), 1, 20, n_or=4, reunit_every=1,
                                storage=12 if nc == 3 else 18, precision=4, hot_start=False)
                cs.wait(jid, 120.0)
                st = cs.status(jid)
                calib[(nc, dims)] = 20 * 5 * 4 * int(np.prod(dims)) / max(st.t_end - st.t_start, 1e-6)
        # steady state of the served engine on the headline lattice: SU(3) 32^4 FP32-12
        # jobs of 40 and 260 iterations, each alone; the difference of their times is
        # the cost of 220 iterations without the job's set-up (table upload, graph
        # capture, start kernels) and retirement, which every job pays once
        times = {}
        for n_it in (40, 260, 40, 260):
            jid = cs.submit(3, (32, 32, 32, 32), 6.0, 2, n_it, n_or=4, reunit_every=1, storage=12, precision=4,
                            hot_start=False)
            cs.wait(jid, 120.0)
            st = cs.status(jid)
            times.setdefault(n_it, []).append(max(st.t_end - st.t_start, 1e-6))
        cs.stop()
    V32 = 32 ** 4
    n_steady = 220
    steady_s = max(min(times[260]) - min(times[40]), 1e-6)
    # HB + 4 OR (9 link transfers per update), reunitarisation (2 per link), plaquette
    # (1) and Polyakov loop (1/4): 48.25 x 4V links of 48 B per iteration
    it_bytes = 4 * V32 * 48 * 48.25
    steady = {"iterations": n_steady, "s": steady_s,
              "link_updates_per_s": n_steady * 5 * 4 * V32 / steady_s,
              "iteration_frac": n_steady * it_bytes / steady_s / (PEAK_HBM_GBS * 1e9),
              "whole_job_260": {"s": min(times[260]),
                                "iteration_frac": 260 * it_bytes / min(times[260]) / (PEAK_HBM_GBS * 1e9)},
              "note": "SU(3) 32^4 FP32-12 jobs alone through the job server (a large-volume group: the "
                      "single-lattice update kernels with the context's launch shapes for 32^4, one launch per "
                      "member, and the fused plaquette + Polyakov measurement, captured in a hipGraph), HB + 4 OR "
                      "+ reunit + plaquette + Polyakov per iteration; 220 iterations = a 260-iteration job minus a "
                      "40-iteration one (best of two each), start to end"}
    # the generation driver on the same lattice description right after those jobs:
    # the device runs ~1% slower a minute into sustained work than at the start of the
    # run, where the headline is measured, so the served figure is set beside the
    # driver's at the same point
    gs = sun_amd.new_stream()
    with sun_amd.Lattice(ctx, 3, (32, 32, 32, 32), 6.0, 12, 4) as gl:
        gl.cold_start(gs)
        gl.generate(seed=2, n_iter=20, n_or=4, reunit_every=1, stream=gs)
        sun_amd.sync(gs)
        t0 = time.perf_counter()
        gl.generate(seed=2, n_iter=n_steady, n_or=4, reunit_every=1, first_sweep=20, stream=gs)
        sun_amd.sync(gs)
        gen_s = time.perf_counter() - t0
    steady["generate_same_point"] = {"s": gen_s,
                                     "iteration_frac": n_steady * it_bytes / gen_s / (PEAK_HBM_GBS * 1e9),
                                     "note": "sun_generate, 220 iterations of the same 32^4 FP32-12 description "
                                             "(context launch shapes), run right after the steady-state jobs"}
    est = [j["n_iter"] * 5 * 4 * int(np.prod(j["dims"])) / calib[(j["nc"], j["dims"])] for j in jobs]
    rate = util / float(np.mean(est))
    gaps = rng.exponential(1.0 / rate, n_jobs)
    updates = sum(j["n_iter"] * 5 * 4 * int(np.prod(j["dims"])) for j in jobs)
    with sun_amd.Server(ctx, budget, max_jobs=256) as srv:
        srv.start()
        ids = []
        t0 = time.perf_counter()
        t_next = 0.0
        for j, g in zip(jobs, gaps):
            t_next += g
            delay = t_next - (time.perf_counter() - t0)
            if delay > 0:
                time.sleep(delay)
            ids.append(srv.submit(j["nc"], j["dims"], j["beta"], j["seed"], j["n_iter"], n_or=4, reunit_every=1,
                                  storage=j["storage"], precision=4, hot_start=j["hot_start"]))
        for jid in ids:
            srv.wait(jid, 600.0)
        srv.stop()
        st = [srv.status(i) for i in ids]
        counters = srv.stats()
    lat = np.array([s.t_end - s.t_submit for s in st])
    queue = np.array([s.t_start - s.t_submit for s in st])
    span = max(s.t_end for s in st) - min(s.t_submit for s in st)
    return {"value": updates / span, "unit": "link-updates/s", "jobs": n_jobs,
            "busy_fraction": counters.busy_s / span,
            "service_model": {f"su{nc}_{dims[0]}^4": round(r / 1e9, 3) for (nc, dims), r in calib.items()},
            "steady_su3_32x4": steady,
            "p50_latency_s": float(np.percentile(lat, 50)), "p99_latency_s": float(np.percentile(lat, 99)),
            "p50_queue_s": float(np.percentile(queue, 50)), "p99_queue_s": float(np.percentile(queue, 99)),
            "span_s": span, "arrival_rate_per_s": rate, "busy_s": counters.busy_s, "steps": int(counters.steps),
            "config": "Poisson arrivals (numpy seed 5) at ~75% load of a measured service-time model "
                      "(service_model: 1e9 link-updates/s per N and volume, one job alone); N in {2,3,4}, volumes "
                      "{8^4,12^4,16^4,24^4,32^4}, beta SU(2) [2.2,2.6], SU(3) [5.6,6.2], SU(4) [10.5,11.2], "
                      "50..500 iterations of HB + 4 OR + reunit + plaquette + Polyakov, FP32 links (SU(3) "
                      "12-real), FP64 reductions, hot/cold 50/50, 64 GiB budget"}


def measurement_leg(sun_amd, ctx, lat, stream):
    """The reference's static-potential chain (test.cpp:170-230) on the generated 32^4
    FP32-12 field: link monitor (before and after a reunitarisation), APE smearing in
    space (w 0.2, 25 steps, 10 hits),
    multihit (100 hits) into an 18-real FP32 lattice, Wilson loops r, T <= 16, and the
    extended multihit (10 heatbath sweeps of every site's 3^3 box of temporal links)."""
    V = int(np.prod(DIMS))
    reps = 20
    # the launch timings before this leg ran sweeps without reunitarisation
    before = lat.link_monitor(stream)
    lat.reunitarize(stream)
    t0 = time.perf_counter()
    for _ in range(reps):
        mon = lat.link_monitor(stream)
    mon_s = (time.perf_counter() - t0) / reps
    t0 = time.perf_counter()
    lat.ape_smear(0.2, 25, 10, 1e-10, stream=stream)
    ape_s = time.perf_counter() - t0
    with sun_amd.Lattice(ctx, 3, DIMS, BETA, 18, 4) as mh:
        t0 = time.perf_counter()
        lat.multihit(mh, 7, 100, stream=stream)
        mh_s = time.perf_counter() - t0
        t0 = time.perf_counter()
        W = mh.wilson_loops(16, 16, stream=stream)
        wl_s = time.perf_counter() - t0
        t0 = time.perf_counter()
        lat.multihit_ext(mh, 7, 10, stream=stream)
        mhx_s = time.perf_counter() - t0
    return {
        "link_monitor": {"ms": mon_s * 1e3, "read_gbs": 4 * V * link_bytes(3, 12, 4) / mon_s / 1e9,
                         "max_unitarity_dev": float(mon[4]), "mean_det": [float(mon[2]), float(mon[3])],
                         "max_unitarity_dev_before_reunit": float(before[4]),
                         "note": "synchronous call (kernel + finalize + 48-byte copy)"},
        "ape_space_25_steps_s": ape_s,
        "multihit_100_hits_s": mh_s,
        "wilson_loops_r16_t16_s": wl_s,
        "multihit_ext_10_hits_s": mhx_s,
        "multihit_ext_link_updates_per_s": 27 * 10 * V / mhx_s,
        "W_r_T4": [float(W[r, 4].real) for r in range(1, 9)],
        "W_r4_T": [float(W[4, t].real) for t in range(1, 9)],
    }


def operator_loops_leg(sun_amd, ctx, stream, calibrate=False):
    """Operator-basis Wilson loops on a 32^4 SU(3) FP64 18-real field (the
    reference's A0 measurement, test.cpp:255-298: Sigma_g_plus(12, 16), r = 2..12,
    the three spatial directions; the 33 family's operator field and correlator at
    r = 12).  Roofline of the correlator: FP64 operations of the traces, V nop^2 (T + 1)
    Frobenius products of 18 reals, over the time of one correlator (its time lines,
    matrix-core kernel and finalize) measured with HIP events on its stream.  calibrate: two plain copies of the 604 MB link field first (the size
    reference for counter passes)."""
    V = int(np.prod(DIMS))
    T = 16
    out = {"lattice": list(DIMS), "precision": "f64", "storage": 18, "rmax": 12, "tmax": T}
    with sun_amd.Lattice(ctx, 3, DIMS, BETA, 18, 8) as lat:
        lat.hot_start(21, stream)
        for it in range(2):
            lat.heatbath(22, it, stream)
            lat.overrelax(stream)
        if calibrate:
            with sun_amd.Lattice(ctx, 3, DIMS, BETA, 18, 8) as tmp:
                for _ in range(2):
                    tmp.copy_from(lat, stream)
                sun_amd.sync(stream)
        t0 = time.perf_counter()
        W = lat.wilson_loops_ops(12, T, sun_amd.WLOP_A0, stream)
        out["a0_measurement_s"] = time.perf_counter() - t0
        out["a0_W00_r4"] = [float(W[2, 0, t]) for t in range(0, 9)]
        for fam, name in ((sun_amd.WLOP_A0, "a0"), (sun_amd.WLOP_33, "f33")):
            with sun_amd.WilsonLoopOps(lat, fam, T) as ops:
                nop = ops.nop
                tm = sun_amd.Timer()
                ops.fields(12, 0, stream)
                ops.correlate(12, 0, stream)
                sun_amd.sync(stream)
                tm.start(stream)
                for _ in range(5):
                    ops.fields(12, 0, stream)
                tm.stop(stream)
                f_ms = tm.ms() / 5
                tm.start(stream)
                for _ in range(5):
                    ops.correlate(12, 0, stream)
                tm.stop(stream)
                c_ms = tm.ms() / 5
                tm.close()
                alg = V * nop * nop * (T + 1) * 36
                tfs = alg / (c_ms * 1e-3) / 1e12
                out[name] = {"nop": nop, "fields_ms_r12": f_ms, "correlate_ms_r12": c_ms,
                             "correlate_roofline": {"bound": "mfma_f64", "achieved": tfs, "peak": PEAK_F64_TFS,
                                                    "unit": "TFLOP/s", "frac": tfs / PEAK_F64_TFS,
                                                    "alg_flops_per_correlator": alg}}
    return out


def kernels_only(sun_amd, large=False, shapes=None, variant=None):
    """For rocprofv3 counter passes.  Default: on the 32^4 FP32 12-real field after
    100 iterations, 2 copies of the field (calibration: a plain copy of known size),
    then 8 overrelaxation launches, 8 heatbath launches, reunitarize, plaquette,
    Polyakov loop.  With large: the same on the 64^4 FP32 8-real field (Haar start,
    beta=6.2) after 20 iterations.  With variant (N, storage, precision): the same at
    32^4 for that kernel variant (beta 2.3 / 6.0 / 11.0 for N = 2 / 3 / 4) after 20
    iterations.  Launch shapes: those of the committed summary (as in the benchmark),
    or with --autotune (and for a variant) the tune cache in $SUN_RESOURCE_PATH
    written by a preceding run with the same variable; without a cache the autotuner
    runs first and its trial launches appear in the profile too."""
    ctx = sun_amd.Context(0, 0, 1)
    nc, prec = 3, 4
    dims, beta, storage = ((64, 64, 64, 64), 6.2, 8) if large else (DIMS, BETA, 12)
    if variant:
        nc, storage, prec = variant
        beta = {2: 2.3, 3: 6.0, 4: 11.0}[nc]
    lat = sun_amd.Lattice(ctx, nc, dims, beta, storage, prec)
    if not variant:
        pin_shapes(lat, shapes)
    tmp = sun_amd.Lattice(ctx, nc, dims, beta, storage, prec)
    s = sun_amd.new_stream()
    if large:
        lat.hot_start(3, s)
    else:
        lat.cold_start(s)
    # iterations first, so clocks are at their sustained level when the launches
    # below run (the profile averages then match the benchmark's timings)
    lat.generate(seed=2, n_iter=20 if (large or variant) else 100, n_or=4, reunit_every=0 if large else 1, stream=s)
    for _ in range(2):
        tmp.copy_from(lat, s)
    for parity in (0, 1):
        for mu in range(4):
            lat.overrelax_sub(parity, mu, s)
    for parity in (0, 1):
        for mu in range(4):
            lat.heatbath_sub(2, 3, parity, mu, s)
    lat.reunitarize(s)
    lat.plaquette(s)
    lat.polyakov(s)
    sun_amd.sync(s)
    print(f"kernels-only: field {lat.bytes} bytes, copy calibration size {tmp.bytes} bytes; shapes: overrelaxation "
          f"{json.dumps(lat.get_launch(1).as_dict())}, heatbath {json.dumps(lat.get_launch(0).as_dict())}")
    tmp.close()
    lat.close()
    ctx.close()


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--no-cpu", action="store_true", help="skip the cpu_baseline leg")
    ap.add_argument("--no-plain", action="store_true", help="skip the plain FP64 GPU leg")
    ap.add_argument("--no-batch", action="store_true", help="skip the batched 64-lattice leg")
    ap.add_argument("--no-large", action="store_true", help="skip the 64^4 FP32 8-real leg")
    ap.add_argument("--no-serve", action="store_true", help="skip the served (Poisson arrivals) leg")
    ap.add_argument("--no-meas", action="store_true", help="skip the smearing / Wilson loop leg")
    ap.add_argument("--serve-jobs", type=int, default=48, help="jobs in the served leg")
    ap.add_argument("--large", action="store_true", help="with --kernels-only: the 64^4 FP32 8-real field")
    ap.add_argument("--variant", default=None,
                    help="with --kernels-only: N,storage,precision of another kernel variant at 32^4 (e.g. 4,18,4)")
    ap.add_argument("--batch-classes", action="store_true",
                    help="only the 64-lattice batch's overrelaxation sweep by volume class (with copy calibration, "
                         "for rocprofv3)")
    ap.add_argument("--ops-only", action="store_true",
                    help="only the operator-basis Wilson loop leg (with copy calibration, for rocprofv3)")
    ap.add_argument("--kernels-only", action="store_true",
                    help="fixed short launch sequence for profiler counter passes (no JSON line)")
    ap.add_argument("--autotune", action="store_true",
                    help="launch shapes from the autotuner instead of those of the committed profiles")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this engine runs on one GPU; --gpus {args.gpus} is not supported "
              "(independent lattices and jobs run one process per GPU without communication)",
              file=sys.stderr)
        sys.exit(2)

    import sun_amd
    shapes32 = None if args.autotune else profiled_shapes(PROFILE_32)
    shapes64 = None if args.autotune else profiled_shapes(PROFILE_64)
    if args.batch_classes:
        ctx = sun_amd.Context(0, 0, 0)
        print(json.dumps(batch_classes(sun_amd, ctx, sun_amd.new_stream(), calibrate=True)))
        ctx.close()
        return
    if args.ops_only:
        ctx = sun_amd.Context(0, 0, 0)
        print(json.dumps(operator_loops_leg(sun_amd, ctx, sun_amd.new_stream(), calibrate=True)))
        ctx.close()
        return
    if args.kernels_only:
        variant = tuple(int(v) for v in args.variant.split(",")) if args.variant else None
        kernels_only(sun_amd, large=args.large, shapes=shapes64 if args.large else shapes32, variant=variant)
        return
    ctx = sun_amd.Context(0, 0, 1)
    V = int(np.prod(DIMS))
    updates_per_step = 5 * 4 * V
    storage, prec = 12, 4
    lat = sun_amd.Lattice(ctx, 3, DIMS, BETA, storage, prec)
    shape_source = pin_shapes(lat, shapes32)
    if shapes32:
        # the same shapes as the context's for this lattice description, so the job
        # server's 32^4 FP32-12 jobs run them too (a tune-cache entry, in effect)
        for kernel, key in ((1, "overrelax"), (0, "heatbath")):
            c = shapes32[key]
            ctx.set_launch(3, DIMS, BETA, storage, prec, kernel, c["block"], tuple(c["brick"]), c["lds"], c["piped"])
    stream = sun_amd.new_stream()
    lat.cold_start(stream)
    sun_amd.sync(stream)

    # warmup (tunes launch shapes, builds and replays the graph)
    lat.generate(seed=2, n_iter=args.warmup, n_or=4, reunit_every=1, first_sweep=0, stream=stream)
    sun_amd.sync(stream)
    t0 = time.perf_counter()
    obs = lat.generate(seed=2, n_iter=args.steps, n_or=4, reunit_every=1, first_sweep=args.warmup, stream=stream)
    sun_amd.sync(stream)
    wall = time.perf_counter() - t0
    value = updates_per_step * args.steps / wall

    # dominant kernel: per-launch durations on the same stream
    or_ms = time_launches(sun_amd, lat, stream, hb=False, reps=64)
    hb_ms = time_launches(sun_amd, lat, stream, hb=True, reps=32)
    launch_or, launch_hb = lat.get_launch(1).as_dict(), lat.get_launch(0).as_dict()
    traffic, traffic_src = profile_traffic(launch_or)
    B = link_bytes(3, storage, prec)
    per_launch = 9 * B * (V // 2)
    or_gbs = per_launch / (or_ms * 1e-3) / 1e9
    hb_gbs = per_launch / (hb_ms * 1e-3) / 1e9
    iter_bytes = 4 * V * B * (45 + 2 + 1 + 0.25)
    step_ms = wall / args.steps * 1e3

    out = {
        "metric": "SU(3) link updates/s + % HBM roofline at 32^4",
        "value": value,
        "unit": "link-updates/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": step_ms,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic (cold start, Philox heatbath)",
        "config": {"workload": "SU(3) 32^4 beta=6.0 cold start, FP32 12-real links; step = 1 heatbath + "
                               "4 overrelaxation sweeps + reunitarize + plaquette + Polyakov (FP64 sums), "
                               "hipGraph replay",
                   "lattice": list(DIMS), "beta": BETA, "storage": storage, "precision": "f32",
                   "updates_per_step": updates_per_step},
        "roofline": {"bound": "hbm", "achieved": or_gbs, "peak": PEAK_HBM_GBS, "unit": "GB/s",
                     "frac": or_gbs / PEAK_HBM_GBS, "traffic": traffic, "traffic_source": traffic_src,
                     "kernel": "overrelaxation (parity, mu) launch",
                     "algorithmic_bytes_per_launch": per_launch, "avg_launch_ms": or_ms,
                     "heatbath_launch_ms": hb_ms, "heatbath_gbs": hb_gbs,
                     "launch_shape": launch_or, "heatbath_launch_shape": launch_hb,
                     "launch_shape_source": shape_source,
                     "iteration_frac": iter_bytes / (step_ms * 1e-3) / 1e9 / PEAK_HBM_GBS},
        "observables": {"plaquette_last": float(obs[-1, :2].mean()), "polyakov_last": [float(obs[-1, 2]),
                                                                                        float(obs[-1, 3])]},
        "device": ctx.device_name(),
    }
    if not args.no_meas:
        out["measurement_chain"] = measurement_leg(sun_amd, ctx, lat, stream)
    lat.close()
    if not args.no_meas:
        out["operator_loops"] = operator_loops_leg(sun_amd, ctx, stream)

    if not args.no_plain:
        out["plain_fp64"] = plain_fp64_leg(sun_amd, ctx, stream, value, updates_per_step)
        out["precision"] = precision_leg(sun_amd, ctx, stream, shapes32)
    if not args.no_large:
        out["large_64x4_f32_8"] = large_leg(sun_amd, ctx, stream, shapes=shapes64)
        out["shard_share_64x4_f32_8"] = shard_leg(sun_amd, ctx, stream)
    if not args.no_batch:
        out["batched"] = batched_leg(sun_amd, ctx, stream)
        out["batched"]["by_volume_class"] = batch_classes(sun_amd, ctx, stream)
    if not args.no_serve:
        out["served"] = served_leg(sun_amd, ctx, args.serve_jobs)
    if not args.no_cpu:
        cb = cpu_baseline()
        out["cpu_baseline"] = cb
        out["gain_vs_cpu"] = value / cb["value"]
    ctx.close()
    print(json.dumps(out))


if __name__ == "__main__":
    main()
