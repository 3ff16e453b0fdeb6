"""Benchmark: batched mixed-precision TDBP of a 27-burst IW scene vs the plain
FP64 kernel, on one MI355X.

Workload (IW scene): 3 subswaths x 9 bursts of uneven size, pulses
U[1350,1550], samples U[18000,25000], output tiles U[1000,4500] x
U[1200,1600] on an fBm DEM (seed 1).  Range-compressed inputs are complex64,
synthesised on the GPU (band-limited circular Gaussian clutter + point
targets) and packed to the storage type on the device; they are resident in
HBM before timing starts.

One step = one batched mixed-precision pass over all 27 bursts (one graph
replay: queue reset, aperture fits, one persistent launch).  The plain FP64
kernel is timed on the same bursts, one launch per burst as the drop-in runs
it.  value = pixel-pulse pairs / step time, in Gpixel*pulse/s.

Prints ONE JSON line.  --gpus N > 1 is rejected: this engine runs on one GPU.
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "Gpixel·pulse/s backprojected, batched mixed vs plain FP64, ≤1 mrad RMS phase"
FLOP_PER_PAIR = 30.0          # algorithmic work per pixel-pulse pair
PEAK_FP32_TFLOPS = 157.3      # MI355X vector FP32
PEAK_FP64_TFLOPS = 78.6       # MI355X vector FP64


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def errors(g, o):
    g = g.astype(np.complex128).ravel()
    o = o.astype(np.complex128).ravel()
    m = np.abs(o) > 0
    g, o = g[m], o[m]
    w = np.abs(o) ** 2
    ph = float(np.sqrt(np.sum(w * np.angle(g * np.conj(o)) ** 2) / np.sum(w)))
    amp = float(np.sqrt(np.sum((np.abs(g) - np.abs(o)) ** 2) / np.sum(w)))
    return ph, amp


def measured_traffic(storage, pairs, variant=None):
    """(HBM bytes per launch, variant measured, unit utilisations) from the
    committed PMC summary (FETCH_SIZE and WRITE_SIZE runs, calibrated by kernels
    of known size; VALU and texture-addresser busy fractions) when it was
    measured on this workload and storage -- the line of `variant` where the
    summary holds one, else its first; else (None, None, None)."""
    import re
    path = os.path.join(ROOT, "profiles", "k_batch_mixed_iw_scene_pmc.md")
    if not os.path.exists(path):
        return None, None, None
    txt = open(path).read()
    lines = re.findall(r"traffic_bytes_per_launch=(\d+) storage=(\w+) variant=(\d+) "
                       r"pairs=(\d+)\s+valu_busy=([\d.]+) ta_busy=([\d.]+) l2_hit=([\d.]+)", txt)
    lines = [m for m in lines if m[1] == storage and int(m[3]) == pairs]
    if not lines:
        return None, None, None
    pick = next((m for m in lines if variant is not None and int(m[2]) == variant), lines[0])
    busy = {"valu": float(pick[4]), "texture_addresser": float(pick[5]),
            "l2_hit_rate": float(pick[6])}
    return int(pick[0]), int(pick[2]), busy


def rc_traffic():
    """HBM bytes per burst of the range compression (cf32 rows; packed words)
    from the committed PMC summary (FETCH_SIZE and WRITE_SIZE runs), or None."""
    import re
    path = os.path.join(ROOT, "profiles", "range_compress_iw_burst_pmc.md")
    if not os.path.exists(path):
        return None
    txt = open(path).read()
    out = {}
    for key in ("cf32", "packed"):
        m = re.search(r"traffic_bytes_per_burst_%s=(\d+)" % key, txt)
        if m:
            out[key] = int(m.group(1))
    return out or None


def cpu_baseline(sc, d_data, budget_s=15.0):
    """The reference CPU pixelint (oracle/_ref, built from the reference's own
    sources) on a bounded row sample of burst 0, all host threads; falls back
    to the oracle restatement when the reference build is absent."""
    from oracle import pyoracle

    g = sc.geom
    data = (d_data.download() if hasattr(d_data, "download") else d_data).reshape(g.L, g.S)
    orc = pyoracle.Oracle()
    kind = "reference" if pyoracle.ref_available() else "port"
    ref = pyoracle.RefCPU() if kind == "reference" else None
    xyz, xyzfit = orc.setxyz(g, sc.dem)
    coef = orc.fitcoef(g, xyzfit)
    azoff = orc.setazoff(g, coef)
    rows = np.nonzero((azoff > 0).any(1))[0]
    mid = rows[len(rows) // 2]
    threads = int(os.environ.get("OMP_NUM_THREADS", "0") or 0) or os.cpu_count()

    def run(r0, r1, lib=None):
        sl = slice(r0, r1)
        t = time.perf_counter()
        if lib is not None:
            lib.pixelint(g, data, sc.satloc, xyz, azoff, rows=sl)
        elif ref is not None:
            ref.pixelint(g, data, sc.satloc, xyz, azoff, rows=sl)
        else:
            orc.pixelint(g, data, sc.satloc, xyz, azoff, semantics=pyoracle.CPU_SEMANTICS,
                         rows=sl)
        dt = time.perf_counter() - t
        a = azoff[sl]
        s = np.floor(a - g.A // 2 + 0.5)      # C round() for positive values
        e = np.minimum(np.floor(a + g.A // 2 + 0.5), g.L - 1)
        pairs = int(np.sum(np.where(a > 0, e - np.maximum(s, 0), 0)))
        return pairs, dt

    pairs, dt = run(mid, mid + 2)                       # calibration
    rate = pairs / max(dt, 1e-6)
    nrows = int(max(2, min(len(rows), budget_s * rate / max(pairs / 2, 1))))
    r0 = max(0, mid - nrows // 2)
    pairs, dt = run(r0, r0 + nrows)
    out = {"value": pairs / dt / 1e9, "unit": "Gpixel·pulse/s", "cores": threads,
           "kind": kind,
           "sample": f"pixelint of burst 0 ({g.L}x{g.S}), window rows {r0}..{r0 + nrows - 1} "
                     f"x {g.demwidth} px, {pairs} pairs in {dt:.1f} s, gcc -O2 -fopenmp, "
                     f"OMP threads {threads}"}
    if ref is not None and pyoracle.ref_available(pyoracle.REF_O0_SO):
        # the same pixelint built without optimisation, as the reference's own
        # build script compiles it (build_proc:10), on a shorter sample
        lib0 = pyoracle.RefCPU(pyoracle.REF_O0_SO)
        p0, t0 = run(mid, mid + 2, lib0)
        n0 = int(max(2, min(len(rows), budget_s / 2 * p0 / max(t0, 1e-6) / max(p0 / 2, 1))))
        a0 = max(0, mid - n0 // 2)
        p0, t0 = run(a0, a0 + n0, lib0)
        out["O0"] = {"value": p0 / t0 / 1e9, "sample": f"window rows {a0}..{a0 + n0 - 1}, "
                     f"{p0} pairs in {t0:.1f} s, gcc -O0 -fopenmp, OMP threads {threads}"}
    return out


def cpu_baseline_entry(sc, data, pairs, td):
    """The reference's whole CPU entry azimuth_compress_cpu_ (oracle/_ref,
    built from its own sources, gcc -O2 -fopenmp) on the same burst, DEM file
    and .geo file as the drop-in: one full call, file I/O included.  None when
    the reference build is absent."""
    import ctypes
    from oracle import pyoracle

    if not pyoracle.ref_available():
        return None
    ref = pyoracle.RefCPU()
    g = sc.geom
    demf, geof = os.path.join(td, "ref.dem"), os.path.join(td, "ref.geo")
    sc.dem.astype(np.int16).tofile(demf)
    np.zeros((sc.demlength, g.demwidth), np.complex64).tofile(geof)
    fdd, fdo = os.open(demf, os.O_RDONLY), os.open(geof, os.O_RDWR)
    threads = int(os.environ.get("OMP_NUM_THREADS", "0") or 0) or os.cpu_count()
    try:
        t = time.perf_counter()
        ref.azimuth_compress_cpu(data, sc.satloc, g.L, g.S, g.demwidth, sc.demlength, fdo, fdd,
                                 g.deltalat, g.deltalon, g.firstlat, g.firstlon, sc.latlons,
                                 g.timeorbit, g.xx, g.vv, g.rngstart, g.rngend, g.tmid,
                                 g.xyz_mid, g.vel_mid, g.dmrg, g.wvl, g.A, g.angc0, g.angc1,
                                 g.prf)
        ctypes.CDLL(None).fflush(None)
        dt = time.perf_counter() - t
    finally:
        os.close(fdd)
        os.close(fdo)
    return {"value": pairs / dt / 1e9, "unit": "Gpixel·pulse/s", "cores": threads,
            "kind": "reference",
            "sample": f"one full azimuth_compress_cpu_ call on the same burst ({g.L}x{g.S} -> "
                      f"{g.nlines}x{g.demwidth} px, {pairs} pairs) and files in {dt:.1f} s, "
                      f"DEM read and .geo read-modify-write included, gcc -O2 -fopenmp, "
                      f"OMP threads {threads}"}


def cpu_baseline_rc(lines, chirp_header, budget_s=10.0):
    """Range compression by the oracle (numpy FFT in FP64, one thread) on a
    bounded sample: the given lines, repeated until about budget_s of work.
    The reference's CPU path (processsub.f90 with FFTW) cannot be built here:
    FFTW is not installed."""
    from oracle import range_oracle as RO

    c = RO.chirp_params(chirp_header)
    done, t0 = 0, time.perf_counter()
    while time.perf_counter() - t0 < budget_s:
        RO.compress(lines, c)
        done += len(lines)
    dt = time.perf_counter() - t0
    return {"value": round(done / dt, 2), "unit": "lines/s", "cores": 1, "kind": "port",
            "sample": f"oracle range compression (numpy FFT, FP64) of {done} lines "
                      f"({len(lines)} distinct) in {dt:.1f} s; the reference's FFTW path "
                      f"is not buildable here"}


def cpu_baseline_igram(img1, img2, rows_total, budget_s=10.0):
    """crossmul by the oracle (numpy, FP64, one thread) on a bounded sample
    of grid rows, repeated until about budget_s of work, scaled to a whole
    interferogram."""
    from oracle import igram_oracle as IO

    done, t0 = 0, time.perf_counter()
    while time.perf_counter() - t0 < budget_s:
        IO.crossmul(img1, img2)
        done += img1.shape[0]
    dt = time.perf_counter() - t0
    return {"value": round(dt / done * rows_total * 1e3, 1), "unit": "ms per interferogram",
            "cores": 1, "kind": "port",
            "sample": f"oracle crossmul (numpy, FP64) of {done} rows x {img1.shape[1]} "
                      f"({img1.shape[0]} distinct) in {dt:.1f} s, scaled to {rows_total} rows"}


def single_burst(args, synth, T):
    """One burst, FP64 kernel vs mixed for each storage type: the full IW burst
    with errors against the FP64 kernel, or the small burst against the FP64
    oracle."""
    from oracle import pyoracle

    full = args.workload == "burst"
    sc = synth.iw_burst() if full else synth.small_burst()
    g = sc.geom
    if full:
        d_data = T.DeviceArray((g.L, g.S), np.complex64)
        d_sat = T.DeviceArray.from_host(sc.satloc)
        synth.device_samples(sc, d_data, d_sat)
    else:
        d_data = T.DeviceArray.from_host(synth.host_samples(sc))
        d_sat = T.DeviceArray.from_host(sc.satloc)
    d_dem = T.DeviceArray.from_host(sc.dem)
    d_coef = T.DeviceArray((g.nlines, 3), np.float64)
    d_out = T.DeviceArray((g.nlines, g.demwidth), np.complex64)
    d_pairs = T.DeviceArray((g.nlines,), np.int64)
    T.fit_aperture(g, d_dem, d_coef)
    T.pair_count(g, d_coef, d_pairs)
    pairs = int(d_pairs.download().sum())
    stream = T.Stream()
    ev0, ev1 = T.Event(), T.Event()

    def timed(smp, prec, reps):
        T.backproject(g, smp, d_sat, d_dem, d_out, prec, d_coef=d_coef, stream=stream)
        stream.sync()
        ev0.record(stream)
        for _ in range(reps):
            T.backproject(g, smp, d_sat, d_dem, d_out, prec, d_coef=d_coef, stream=stream)
        ev1.record(stream)
        stream.sync()
        return ev0.elapsed_ms(ev1) / reps, d_out.download()

    plain_ms, plain = timed(T.samples(d_data), T.PLAIN_FP64, max(2, args.steps // 4))
    if not full:
        ref = pyoracle.Oracle().backproject(g, d_data.download(), sc.satloc, sc.dem)[0]
        against = "FP64 oracle (reference GPU semantics)"
    else:
        ref = plain
        against = "FP64 kernel"
    m = ref != 0
    res = {"plain_fp64": {"gpps": round(pairs / plain_ms / 1e6, 2), "ms": round(plain_ms, 4),
                          "vs_reference": dict(zip(("phase_mrad", "amp_rel"),
                                               (lambda e: (round(e[0] * 1e3, 6), e[1]))(
                                                   errors(plain[m], ref[m]))))}}
    for name, dt in (("cf32", T.CF32), ("ci16", T.CI16), ("cf16", T.CF16), ("cbf16", T.CBF16)):
        if dt == T.CF32:
            smp = T.samples(d_data)
        else:
            pk, scl = T.pack(d_data, g.L, g.S, dt)
            smp = T.samples(pk, dt, scl)
        ms, out = timed(smp, T.MIXED, args.steps)
        ph, amp = errors(out[m], ref[m])
        res["mixed_" + name] = {"gpps": round(pairs / ms / 1e6, 2), "ms": round(ms, 4),
                                "phase_mrad": round(ph * 1e3, 5), "amp_rel": amp,
                                "meets_bar": bool(ph <= 1e-3 and amp <= 1e-4),
                                "speedup_vs_plain": round(plain_ms / ms, 3)}
        log(f"mixed {name}: {ms:.3f} ms ({pairs / ms / 1e6:.1f} GP/s), phase {ph * 1e3:.4f} "
            f"mrad, amp {amp:.2e}")
    best = res["mixed_cf32"]
    cpu = None if args.no_cpu else cpu_baseline(sc, d_data)
    line = {"metric": METRIC, "value": best["gpps"], "unit": "Gpixel·pulse/s", "n_gpus": 1,
            "steps": args.steps, "warmup": 1, "ms_per_step": best["ms"],
            "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
            "dtype": "f32 (f64 per-tile reference)", "data": "synthetic",
            "config": {"workload": (
                "one IW burst 1500 x 21000 -> 4000 x 1500 px, fBm DEM" if full else
                "512 x 4096 burst -> 256 x 256 px, flat DEM, A=256"),
                "pairs": pairs, "errors_against": against,
                "storage": "cf32 (value); the packed storages reported beside it, packed "
                           "outside the timed region"},
            "results": res, "cpu_baseline": cpu}
    print(json.dumps(line), flush=True)


def dropin_bench(args, synth, T):
    """The drop-in entry end to end on one IW burst (1500 x 21000 -> 4000 x
    1500 px): burst and pulse positions in host memory, DEM and .geo as files
    (page cache), FP64, mixed cf32 (the value) and mixed cf16.  Rate = pairs /
    wall time of the call,
    host-device copies and file read-modify-write included."""
    import tempfile
    from srg_amd import dropin

    sc = synth.iw_burst()
    g = sc.geom
    d_data = T.DeviceArray((g.L, g.S), np.complex64)
    d_sat = T.DeviceArray.from_host(sc.satloc)
    synth.device_samples(sc, d_data, d_sat)
    data = d_data.download()
    d_dem = T.DeviceArray.from_host(sc.dem)
    d_coef = T.DeviceArray((g.nlines, 3), np.float64)
    d_pairs = T.DeviceArray((g.nlines,), np.int64)
    T.fit_aperture(g, d_dem, d_coef)
    T.pair_count(g, d_coef, d_pairs)
    pairs = int(d_pairs.download().sum())
    call = dropin.BurstCall.from_burst(data, g, sc.satloc, sc.demlength, g.firstlat,
                                       sc.latlons)
    res = {}
    with tempfile.TemporaryDirectory() as td:
        demf, geof = os.path.join(td, "elevation.dem"), os.path.join(td, "scene.geo")
        sc.dem.astype(np.int16).tofile(demf)
        np.zeros((sc.demlength, g.demwidth), np.complex64).tofile(geof)
        fdd, fdo = os.open(demf, os.O_RDONLY), os.open(geof, os.O_RDWR)
        try:
            for name in ("fp64", "mixed_cf32", "mixed_fp16"):
                os.environ["TDBP_PRECISION"] = name
                for _ in range(args.warmup):
                    call.call(fdo, fdd)
                walls, phases = [], []
                for _ in range(args.steps):
                    t0 = time.perf_counter()
                    call.call(fdo, fdd)
                    walls.append((time.perf_counter() - t0) * 1e3)
                    phases.append(dropin.last_timing())
                ms = float(np.median(walls))
                ph = {k: round(float(np.median([p[k] for p in phases])), 3)
                      for k in dropin.TIMING_NAMES}
                # the same calls with TDBP_DROPIN_ASYNC=1: .geo writes overlap the
                # next burst's upload; timed to the last flush
                os.environ["TDBP_DROPIN_ASYNC"] = "1"
                t0 = time.perf_counter()
                for _ in range(args.steps):
                    call.call(fdo, fdd)
                dropin.flush()
                ams = (time.perf_counter() - t0) * 1e3 / args.steps
                os.environ.pop("TDBP_DROPIN_ASYNC", None)
                # TDBP_BATCH=1: the calls stage their bursts; the flush runs them as
                # one batch with one .geo read-merge-write; timed to the flush
                os.environ["TDBP_BATCH"] = "1"
                t0 = time.perf_counter()
                for _ in range(args.steps):
                    call.call(fdo, fdd)
                dropin.flush()
                bms = (time.perf_counter() - t0) * 1e3 / args.steps
                os.environ.pop("TDBP_BATCH", None)
                res[name] = {"gpps_end_to_end": round(pairs / ms / 1e6, 2),
                             "ms_per_call": round(ms, 3), "phases_ms": ph,
                             "async_ms_per_call": round(ams, 3),
                             "async_gpps_end_to_end": round(pairs / ams / 1e6, 2),
                             "deferred_ms_per_call": round(bms, 3),
                             "deferred_gpps_end_to_end": round(pairs / bms / 1e6, 2)}
                log(f"drop-in {name}: {ms:.2f} ms/call ({pairs / ms / 1e6:.1f} GP/s end to "
                    f"end); async {ams:.2f} ms/call ({pairs / ams / 1e6:.1f} GP/s); "
                    f"deferred {bms:.2f} ms/call ({pairs / bms / 1e6:.1f} GP/s); phases {ph}")
            # the CPU twin's entry (azimuth_compress_cpu_): the same burst with the
            # twin's arithmetic (FP64 lerp, unscaled, integer-abs merge)
            os.environ["TDBP_PRECISION"] = "fp64"
            for _ in range(args.warmup):
                call.call(fdo, fdd, entry="cpu")
            walls = []
            for _ in range(args.steps):
                t0 = time.perf_counter()
                call.call(fdo, fdd, entry="cpu")
                walls.append((time.perf_counter() - t0) * 1e3)
            ms = float(np.median(walls))
            res["cpu_twin_fp64"] = {"gpps_end_to_end": round(pairs / ms / 1e6, 2),
                                    "ms_per_call": round(ms, 3)}
            log(f"drop-in azimuth_compress_cpu_ fp64: {ms:.2f} ms/call "
                f"({pairs / ms / 1e6:.1f} GP/s end to end)")
        finally:
            os.environ.pop("TDBP_PRECISION", None)
            os.environ.pop("TDBP_DROPIN_ASYNC", None)
            os.environ.pop("TDBP_BATCH", None)
            os.close(fdd)
            os.close(fdo)
        cpu = None if args.no_cpu else cpu_baseline_entry(sc, data, pairs, td)
    best = res["mixed_cf32"]
    if cpu is None and not args.no_cpu:
        cpu = cpu_baseline(sc, data)
    line = {"metric": METRIC + " (drop-in, end to end)", "value": best["gpps_end_to_end"],
            "unit": "Gpixel·pulse/s", "n_gpus": 1, "steps": args.steps,
            "warmup": args.warmup, "ms_per_step": best["ms_per_call"],
            "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
            "dtype": "f32 (f64 per-tile reference)", "data": "synthetic",
            "config": {"workload": "azimuth_compress_ on one IW burst 1500 x 21000 -> "
                                   "4000 x 1500 px, host buffers, DEM/.geo files",
                       "pairs": pairs},
            "results": res, "cpu_baseline": cpu}
    print(json.dumps(line), flush=True)


def rc_bench(args, synth, T):
    """Range compression of one IW burst on the device (1500 decoded lines of
    30000 samples, IW1 chirp of 3372 samples, 24400 echo samples -> 21028
    compressed) into cf32 rows (the value), and into packed cf16 / ci16 words
    beside it, then the mixed backprojection of the cf32 rows onto 4000 x 1500
    px: raw echoes to image."""
    from srg_amd import raw

    h = raw.header_bytes(raw.IW1)
    c = T.chirp_decode(h)
    S = c.nvalid + 10
    src = synth.fbm_surface((2048, 2048), seed=7)
    sc = synth.make_burst(1500, S, 4000, 1500, dem="fbm", dem_source=src, ntargets=5,
                          clutter_sigma=0.0, seed=0)
    g = sc.geom
    d_raw = T.DeviceArray((g.L, raw.RAW_STRIDE), np.complex64)
    raw.device_lines(sc, c, h, d_raw, noise=0.1, seed=3)
    pw = T.DeviceArray((g.L, S), np.uint32)
    ps = T.DeviceArray((g.L,), np.float32)
    cf = T.DeviceArray((g.L, S), np.complex64)
    d_sat = T.DeviceArray.from_host(sc.satloc)
    d_dem = T.DeviceArray.from_host(sc.dem)
    d_coef = T.DeviceArray((g.nlines, 3), np.float64)
    d_pairs = T.DeviceArray((g.nlines,), np.int64)
    out = T.DeviceArray((g.nlines, g.demwidth), np.complex64)
    T.fit_aperture(g, d_dem, d_coef)
    T.pair_count(g, d_coef, d_pairs)
    pairs = int(d_pairs.download().sum())
    stream = T.Stream()
    ev0, ev1 = T.Event(), T.Event()

    def timed(fn, reps):
        fn()
        stream.sync()
        ev0.record(stream)
        for _ in range(reps):
            fn()
        ev1.record(stream)
        stream.sync()
        return ev0.elapsed_ms(ev1) / reps

    packed = lambda: T.range_compress(d_raw, c, None, packed=(T.CF16, pw, ps),  # noqa: E731
                                      stream=stream)
    both = lambda: T.range_compress(d_raw, c, cf, packed=(T.CF16, pw, ps),  # noqa: E731
                                    stream=stream)
    tdbp_ = lambda: T.backproject(g, T.samples(pw, T.CF16, ps), d_sat, d_dem, out,  # noqa: E731
                                  T.MIXED, d_coef=d_coef, stream=stream)
    def cf32_into(buf, s_):
        T.range_compress(d_raw, c, buf, stream=s_, zero_header=True)

    def packed_into(dt, w_, sc_, s_):
        T.range_compress(d_raw, c, None, packed=(dt, w_, sc_), stream=s_)

    def bp_from(buf, o_, s_):
        T.backproject(g, T.samples(buf), d_sat, d_dem, o_, T.MIXED, d_coef=d_coef, stream=s_)

    ms_cf32 = timed(lambda: cf32_into(cf, stream), args.steps)
    ms_packed = {name: timed(lambda dt=dt: packed_into(dt, pw, ps, stream), args.steps)
                 for name, dt in (("cf16", T.CF16), ("ci16", T.CI16))}
    ms_both = timed(lambda: T.range_compress(d_raw, c, cf, packed=(T.CF16, pw, ps),
                                             stream=stream), max(2, args.steps // 2))
    ms_bp = timed(lambda: bp_from(cf, out, stream), args.steps)
    ms_e2e = timed(lambda: (cf32_into(cf, stream), bp_from(cf, out, stream)), args.steps)

    # A stream of bursts: range compression of burst k+1 (its FFTs) on one
    # stream while burst k is backprojected on the other.  Each stream has
    # its own cf32 rows and image; wall time over nburst bursts.
    cf2 = T.DeviceArray((g.L, S), np.complex64)
    out2 = T.DeviceArray((g.nlines, g.demwidth), np.complex64)
    stream2 = T.Stream()
    bufs = [(stream, cf, out), (stream2, cf2, out2)]

    def burst_stream(nburst, nstreams):
        for k in range(nburst):
            s_, b_, o_ = bufs[k % nstreams]
            cf32_into(b_, s_)
            bp_from(b_, o_, s_)

    nburst = 12
    ms_stream = {}
    for nst in (1, 2):
        best = 1e30
        for _ in range(3):
            T.sync()
            t0 = time.perf_counter()
            burst_stream(nburst, nst)
            stream.sync()
            stream2.sync()
            best = min(best, (time.perf_counter() - t0) * 1e3 / nburst)
        ms_stream[nst] = best
    log(f"burst stream of {nburst}: {ms_stream[1]:.3f} ms/burst on one stream, "
        f"{ms_stream[2]:.3f} on two (compression overlapping backprojection)")
    # Batched: nb bursts range-compressed into their own cf32 rows, then one
    # persistent batch backprojects all of them (process_raw_bursts_batched's
    # launch shape); HIP events around compression + batch, per burst.
    nb = 8
    cfs = [T.DeviceArray((g.L, S), np.complex64) for _ in range(nb)]
    outs = [T.DeviceArray((g.nlines, g.demwidth), np.complex64) for _ in range(nb)]
    bb = T.Batch(T.MIXED, -1)
    for k in range(nb):
        bb.add(g, T.samples(cfs[k]), d_sat, d_dem, outs[k])

    def batched():
        for k in range(nb):
            cf32_into(cfs[k], stream)
        bb.run(stream)

    ms_batched = timed(batched, 3) / nb
    log(f"batched raw -> image over {nb} bursts: {ms_batched:.3f} ms/burst "
        f"({pairs / ms_batched / 1e6:.1f} GP/s), variant {bb.variant}")
    bb.close()
    del cfs, outs
    alg = g.L * ((c.nsamps + 10) * 8 + S * 8)          # read echoes, write cf32 rows
    n_os = 8192
    blocks = g.L * -(-c.nvalid // (n_os - c.npts + 1))
    fft_flop = blocks * (2 * 5 * n_os * 13 + 6 * n_os)  # two transforms + the product
    alg_packed = g.L * ((c.nsamps + 10) * 8 + S * 4 + 4)
    gbps = alg / (ms_cf32 * 1e-3) / 1e9
    img = out.download()
    foc = [abs(np.angle(img[r, col] * np.conj(a))) for (r, col), a in
           zip(sc.targets_px, sc.targets_amp)]
    cpu = None if args.no_cpu else cpu_baseline_rc(d_raw.rows(0, 256).download(), h)
    log(f"range compression (cf32 rows): {ms_cf32:.3f} ms/burst ({g.L / ms_cf32 * 1e3:.0f} "
        f"lines/s, {gbps:.0f} GB/s algorithmic); packed cf16 {ms_packed['cf16']:.3f} ms, ci16 "
        f"{ms_packed['ci16']:.3f} ms; cf32 + cf16 {ms_both:.3f} ms; backprojection (cf32) "
        f"{ms_bp:.3f} ms; raw -> image {ms_e2e:.3f} ms; target phase errors (rad) "
        f"{[round(float(x), 4) for x in foc]}")
    traffic = rc_traffic()
    line = {"metric": "range-compressed lines/s (32768-point matched filter, cf32 output)",
            "value": round(g.L / ms_cf32 * 1e3, 1), "unit": "lines/s", "n_gpus": 1,
            "steps": args.steps, "warmup": 1, "ms_per_step": round(ms_cf32, 4),
            "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
            "dtype": "f32", "data": "synthetic (GPU-generated chirp echoes of 5 targets + noise)",
            "config": {"workload": f"one IW burst: {g.L} decoded lines x 30000 samples, IW1 chirp "
                                   f"{c.npts} samples, {c.nsamps} echo -> {c.nvalid} compressed "
                                   f"(cf32 rows, header zeroed); then mixed backprojection of "
                                   f"the cf32 rows onto 4000 x 1500 px",
                       "pairs": pairs},
            "roofline": {"bound": "valu", "achieved": round(fft_flop / (ms_cf32 * 1e-3) / 1e12, 3),
                         "peak": PEAK_FP32_TFLOPS, "unit": "TFLOP/s",
                         "frac": round(fft_flop / (ms_cf32 * 1e-3) / 1e12 / PEAK_FP32_TFLOPS, 4),
                         "flop_per_burst": fft_flop,
                         "flop_definition": "per 8192-sample block: two transforms of "
                                            "5 N log2 N flop and the 6 N flop spectrum "
                                            "product",
                         "hbm": {"achieved": round(gbps, 1), "peak": 8000.0, "unit": "GB/s",
                                 "frac": round(gbps / 8000.0, 4)},
                         "traffic": traffic.get("cf32") if traffic else None,
                         "algorithmic_bytes_per_burst": alg,
                         "kernel": "k_rc_os (overlap-save FFT pair in LDS)"},
            "packed": {name: {"ms_per_burst": round(ms, 4),
                              "lines_per_s": round(g.L / ms * 1e3, 1),
                              "algorithmic_bytes_per_burst": alg_packed,
                              "traffic": traffic.get("packed") if traffic else None}
                       for name, ms in ms_packed.items()},
            "ms_cf32_and_cf16": round(ms_both, 4),
            "ms_backprojection": round(ms_bp, 4),
            "ms_raw_to_image": round(ms_e2e, 4),
            "raw_to_image_gpps": round(pairs / ms_e2e / 1e6, 2),
            "raw_to_image_batched": {"bursts": nb, "ms_per_burst": round(ms_batched, 4),
                                     "gpps": round(pairs / ms_batched / 1e6, 2)},
            "burst_stream": {"bursts": nburst,
                             "ms_per_burst_one_stream": round(ms_stream[1], 4),
                             "ms_per_burst_two_streams": round(ms_stream[2], 4),
                             "gpps_two_streams": round(pairs / ms_stream[2] / 1e6, 2)},
            "target_phase_err_rad": [round(float(x), 5) for x in foc],
            "cpu_baseline": cpu}
    print(json.dumps(line), flush=True)


def stack_bench(args, synth, T):
    """Time-series stack: 30 acquisitions x 9 uneven bursts onto one common
    13500 x 4000 grid, mixed precision on --storage samples (default cf32),
    admitted into HBM-sized batches,
    each batch one persistent launch plus the device .geo merges; per
    acquisition the merged grid is compared with the FP64 kernel's."""
    from srg_amd import stack as ST

    t0 = time.time()
    stk = synth.ts_stack(nacq=args.acqs)
    grid = stk.grid
    nacq = len(stk.bursts)
    log(f"stack geometry: {nacq} acquisitions, {sum(len(r) for r in stk.bursts)} bursts, "
        f"{time.time() - t0:.1f} s")
    d_dem = T.DeviceArray.from_host(grid.dem)
    bursts = [ST.StackBurst(a, sc.geom, sc.satloc,
                            d_dem.rows(sc.geom.firstline, sc.geom.nlines), payload=sc)
              for a, k, sc in stk.items()]
    g_mixed = [T.DeviceArray((grid.lines, grid.W), np.complex64) for _ in range(nacq)]
    g_fp64 = [T.DeviceArray((grid.lines, grid.W), np.complex64) for _ in range(nacq)]
    for x in g_mixed + g_fp64:
        x.zero()
    maxls = max(b.geom.L * b.geom.S for b in bursts)
    maxnl = max(b.geom.nlines for b in bursts)
    staging = T.DeviceArray((maxls,), np.complex64) if args.storage != "cf32" else None
    out64 = T.DeviceArray((maxnl, grid.W), np.complex64)
    coef = T.DeviceArray((maxnl, 3), np.float64)
    stream = T.Stream()
    e0, e1 = T.Event(), T.Event()
    plain = {"ms": 0.0}

    cpu = {}

    dt = {"cf32": T.CF32, "ci16": T.CI16, "cf16": T.CF16, "cbf16": T.CBF16}[args.storage]

    def loader(i, b, r):
        # Synthesise cf32 samples (into the resident buffer for cf32 storage),
        # run the FP64 kernel on them into the FP64 grids (timed per launch),
        # then pack the resident copy of a packed storage.
        g = b.geom
        stg = r.buffers[0] if dt == T.CF32 else staging.rows(0, g.L * g.S)
        synth.device_samples(b.payload, stg, r.sat, stream=stream)
        if i == 0 and not args.no_cpu:
            stream.sync()
            cpu["bp"] = cpu_baseline(b.payload, stg, budget_s=10.0)
        o = out64.rows(0, g.nlines)
        c = coef.rows(0, g.nlines)
        T.fit_aperture(g, b.dem, c, stream=stream)
        e0.record(stream)
        T.backproject(g, T.samples(stg), r.sat, b.dem, o, T.PLAIN_FP64, d_coef=c,
                      stream=stream)
        e1.record(stream)
        T.merge_geo(g_fp64[b.acq], g.firstline, o, stream=stream)
        if dt != T.CF32:
            T.pack_into(stg, g.L, g.S, dt, r.buffers[0], r.buffers[1], stream=stream)
        stream.sync()
        plain["ms"] += e0.elapsed_ms(e1)

    budget = int(args.hbm_budget * 2**30) if args.hbm_budget else None
    run = ST.run_stack(bursts, g_mixed, loader, precision=T.MIXED, dtype=dt,
                       budget=budget, repeats=args.warmup + args.steps, autotune_reps=2)
    tuned = {"variant": run.tuned[0]} if run.tuned else {}
    if run.tuned:
        log(f"batch autotune: variant {run.tuned[0]}; "
            f"ms per variant {[round(x, 1) for x in run.tuned[1]]}")
    pairs = sum(run.pairs)
    per_batch = [float(np.mean(ms[args.warmup:])) for ms in run.run_ms]
    step_ms = sum(per_batch)
    gpps = pairs / step_ms / 1e6
    plain_gpps = pairs / plain["ms"] / 1e6
    log(f"{len(run.batches)} batch(es), pairs {pairs}: {step_ms:.1f} ms/step "
        f"({gpps:.1f} GP/s); FP64 kernel per burst {plain['ms']:.1f} ms ({plain_gpps:.1f} GP/s)")
    per_acq = []
    for a in range(nacq):
        e = T.compare(g_mixed[a], g_fp64[a])
        per_acq.append(e)
    ph = [e["phase_rms"] * 1e3 for e in per_acq]
    amp = [e["amp_rms"] for e in per_acq]
    log(f"per-acquisition phase vs FP64 (mrad): max {max(ph):.4f} mean {np.mean(ph):.4f}; "
        f"amp max {max(amp):.2e}")

    # Interferograms of consecutive acquisitions on the merged grids, where the
    # stack left them (int/crossmul.f90 with its defaults: scale 1, mask on).
    igram = None
    if nacq > 1 and args.igram_looks > 0:
        lk = args.igram_looks
        T.sync()
        ev_i0, ev_i1 = T.Event(), T.Event()
        ig_ms = []
        oshape = (grid.lines // lk, grid.W // lk)
        ig_out = (T.DeviceArray(oshape, np.complex64), T.DeviceArray(oshape, np.complex64))
        for a in range(nacq - 1):
            ev_i0.record(stream)
            T.crossmul(g_mixed[a], g_mixed[a + 1], looksac=lk, looksdn=lk, stream=stream,
                       out=ig_out)
            ev_i1.record(stream)
            stream.sync()
            ig_ms.append(ev_i0.elapsed_ms(ev_i1))
        del ig_out
        ms_pair = float(np.median(ig_ms[1:] if len(ig_ms) > 1 else ig_ms))
        px = grid.lines * grid.W
        cpu_ig = None
        if not args.no_cpu:
            rows = min(256, grid.lines)
            r0 = stk.bursts[0][0].geom.firstline + 200
            cpu_ig = cpu_baseline_igram(g_mixed[0].rows(r0, rows).download(),
                                        g_mixed[1].rows(r0, rows).download(), grid.lines)
        igram = {"pairs": nacq - 1, "looks": [lk, lk], "ms_per_interferogram": round(ms_pair, 3),
                 "cpu_baseline": cpu_ig,
                 "input_gpx_per_s": round(px / ms_pair / 1e6, 2),
                 "hbm_gbps_algorithmic": round((2 * px * 8 + 2 * px * 8 / lk / lk) / ms_pair / 1e6,
                                               1)}
        log(f"interferograms: {ms_pair:.2f} ms per {grid.lines} x {grid.W} pair "
            f"(looks {lk}x{lk})")
    line = {
        "metric": METRIC, "value": round(gpps, 2), "unit": "Gpixel·pulse/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(step_ms, 3),
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "f32 (f64 per-tile reference)",
        "data": "synthetic (GPU-generated band-limited clutter + point targets, fBm DEM)",
        "config": {"workload": f"time-series stack: {nacq} acquisitions x 9 uneven bursts -> "
                               f"one {grid.lines} x {grid.W} grid, {args.storage}, .geo merge "
                               f"on device",
                   "bursts": len(bursts), "pairs_per_step": pairs,
                   "batches": len(run.batches),
                   "batch_sizes": [len(b) for b in run.batches],
                   "budget_bytes": budget, "variant": tuned.get("variant")},
        "plain_fp64": {"value": round(plain_gpps, 2), "ms_per_pass": round(plain["ms"], 3),
                       "launch": "one per burst"},
        "speedup_vs_plain_fp64": round(plain["ms"] / step_ms, 3),
        "error_vs_fp64_per_acquisition": {
            "phase_mrad_rms": [round(x, 5) for x in ph],
            "amp_rel_rms": [float(f"{x:.3e}") for x in amp],
            "phase_mrad_max": round(max(ph), 5), "amp_rel_max": max(amp),
            "meets_bar": bool(max(ph) <= 1.0 and max(amp) <= 1e-4),
            "extra_nonzero_pixels": sum(e["extra_nonzero"] for e in per_acq)},
        "baselines_m": [round(float(x), 2) for x in np.linalg.norm(stk.baselines, axis=1)],
        "interferograms": igram,
        "cpu_baseline": cpu.get("bp"),
    }
    print(json.dumps(line), flush=True)


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--storage", default="cf32", choices=["cf32", "ci16", "cf16", "cbf16"],
                    help="sample storage of the timed batch (default cf32, the storage that "
                         "meets 1 mrad / 1e-4 against FP64; the others are reported beside it)")
    ap.add_argument("--bursts", type=int, default=27)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--variant", type=int, default=-1,
                    help="kernel variant of the batched mixed run (default: autotune; 8 = MFMA)")
    ap.add_argument("--plain-passes", type=int, default=2)
    ap.add_argument("--workload", default="scene",
                    choices=["scene", "burst", "small", "stack", "dropin", "rc"],
                    help="scene: batched 27-burst IW scene (the headline); burst: one full "
                         "IW burst, plain vs mixed per storage type; small: the 512 x 4096 "
                         "-> 256 x 256 burst per storage type against the FP64 oracle; "
                         "stack: 30 acquisitions x 9 bursts onto one 13500 x 4000 grid; "
                         "dropin: azimuth_compress_ end to end on one IW burst; rc: range "
                         "compression of one IW burst and raw -> image")
    ap.add_argument("--acqs", type=int, default=30, help="stack: acquisitions")
    ap.add_argument("--igram-looks", type=int, default=1,
                    help="stack: looks of the consecutive-pair interferograms (0: none)")
    ap.add_argument("--hbm-budget", type=float, default=0.0,
                    help="stack: admission budget in GiB (default: free HBM less a reserve)")
    ap.add_argument("--profile", action="store_true",
                    help="counter-collection run: a 1 GiB fill and a 1 GiB copy kernel "
                         "(calibration of WRITE_SIZE / FETCH_SIZE) then two eager launches "
                         "of the batched mixed kernel; prints the pairs per launch")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py runs on one GPU only (asked for {args.gpus}); each burst is an "
              f"independent unit and multi-GPU sharding is not part of this build",
              file=sys.stderr)
        sys.exit(2)

    from srg_amd import synth
    from srg_amd import tdbp as T

    T.init(0)
    if args.workload in ("burst", "small"):
        return single_burst(args, synth, T)
    if args.workload == "stack":
        return stack_bench(args, synth, T)
    if args.workload == "dropin":
        return dropin_bench(args, synth, T)
    if args.workload == "rc":
        return rc_bench(args, synth, T)
    t0 = time.time()
    nsub = 3 if args.bursts >= 3 else 1
    scenes = synth.iw_scene(seed=1, nsub=nsub, nburst=max(1, args.bursts // nsub))
    log(f"IW scene geometry: {len(scenes)} bursts in {time.time() - t0:.1f} s")
    dts = {"cf32": T.CF32, "ci16": T.CI16, "cf16": T.CF16, "cbf16": T.CBF16}
    stor = dts[args.storage]

    dev = []
    for sc in scenes:
        g = sc.geom
        d = {"sc": sc,
             "data": T.DeviceArray((g.L, g.S), np.complex64),
             "sat": T.DeviceArray.from_host(sc.satloc),
             "dem": T.DeviceArray.from_host(sc.dem),
             "coef": T.DeviceArray((g.nlines, 3), np.float64),
             "out": T.DeviceArray((g.nlines, g.demwidth), np.complex64),
             "ref": T.DeviceArray((g.nlines, g.demwidth), np.complex64)}
        synth.device_samples(sc, d["data"], d["sat"])
        d["packed"] = {T.CF32: (d["data"], None)}
        for dt in (T.CI16, T.CF16, T.CBF16):
            d["packed"][dt] = T.pack(d["data"], g.L, g.S, dt)
        T.fit_aperture(g, d["dem"], d["coef"])
        dev.append(d)
    T.sync()
    log(f"bursts synthesised and packed on the GPU, {time.time() - t0:.1f} s")

    def smp(d, dt):
        data, scale = d["packed"][dt]
        return T.samples(data, dt, scale)

    if args.profile:
        os.environ["TDBP_GRAPH"] = "0"   # eager dispatches, one per kernel
        nbytes = 1 << 30
        a = T.DeviceArray((nbytes,), np.uint8)
        b = T.DeviceArray((nbytes,), np.uint8)
        a.zero()
        T.check(T.lib().tdbp_dev_copy(b.ptr, a.ptr, nbytes, None))
        T.sync()
        batch = T.Batch(T.MIXED, int(os.environ.get("TDBP_VARIANT", "5")))
        for d in dev:
            batch.add(d["sc"].geom, smp(d, stor), d["sat"], d["dem"], d["out"])
        batch.run()
        batch.run()
        T.sync()
        print(json.dumps({"profile": True, "copy_bytes": nbytes, "pairs_per_launch": batch.pairs,
                          "variant": batch.variant, "storage": args.storage}), flush=True)
        batch.close()
        return

    # The mixed kernel's tile shape: the variant given, or the batch
    # autotuner's pick (every VALU variant timed on this batch of bursts; it
    # also becomes the default of the other-storage batches below).
    if args.variant >= 0:
        T.lib().tdbp_set_variant(args.variant)
        log(f"variant {args.variant} {T.variant_info(args.variant)} (given)")

    ev0, ev1 = T.Event(), T.Event()
    stream = T.Stream()

    # Plain FP64: one launch per burst (the drop-in's way); its outputs are the
    # accuracy reference.
    def plain_pass():
        for d in dev:
            T.backproject(d["sc"].geom, smp(d, T.CF32), d["sat"], d["dem"], d["ref"],
                          T.PLAIN_FP64, d_coef=d["coef"], stream=stream)

    plain_pass()
    stream.sync()
    ev0.record(stream)
    for _ in range(args.plain_passes):
        plain_pass()
    ev1.record(stream)
    stream.sync()
    plain_ms = ev0.elapsed_ms(ev1) / args.plain_passes

    # Batched mixed precision, one graph replay per step.
    batches = {}

    def make_batch(dt):
        b = T.Batch(T.MIXED, -1)
        for d in dev:
            b.add(d["sc"].geom, smp(d, dt), d["sat"], d["dem"], d["out"])
        return b

    batch = make_batch(stor)
    if args.variant < 0:
        best, tune_ms = batch.autotune(reps=2)
        T.lib().tdbp_set_variant(best)   # the other-storage batches below use it too
        log(f"batch autotune: variant {best} {T.variant_info(batch.variant)}; "
            f"ms per variant {[round(x, 2) for x in tune_ms]}")
    batch.run(stream)
    stream.sync()
    pairs = batch.pairs
    for _ in range(args.warmup):
        batch.run(stream)
    stream.sync()
    ev0.record(stream)
    for _ in range(args.steps):
        batch.run(stream)
    ev1.record(stream)
    stream.sync()
    mixed_ms = ev0.elapsed_ms(ev1) / args.steps
    mixed_gpps = pairs / mixed_ms / 1e6
    plain_gpps = pairs / plain_ms / 1e6
    log(f"pairs {pairs}: mixed {args.storage} {mixed_ms:.2f} ms/step ({mixed_gpps:.1f} GP/s), "
        f"plain FP64 {plain_ms:.2f} ms ({plain_gpps:.1f} GP/s)")

    # Accuracy of the timed mixed outputs against the FP64 kernel's images
    # (device error sums per burst, combined by the reference power).
    def scene_error():
        ph2, amp2, wsum = 0.0, 0.0, 0.0
        for d in dev:
            e = T.compare(d["out"], d["ref"], stream=stream)
            ph2 += e["phase_rms"] ** 2 * e["sum_w"]
            amp2 += e["amp_rms"] ** 2 * e["sum_w"]
            wsum += e["sum_w"]
        return float(np.sqrt(ph2 / wsum)), float(np.sqrt(amp2 / wsum))

    ph, amp = scene_error()
    log(f"mixed {args.storage} vs FP64 kernel: phase {ph * 1e3:.4f} mrad, amp {amp:.2e}")

    # End to end from cf32 samples resident in HBM: per step every burst is
    # packed to the storage type (k_pack_scale + k_pack into the buffers the
    # batch reads), then the batch runs.
    e2e = None
    if stor != T.CF32:
        def e2e_step():
            for d in dev:
                g = d["sc"].geom
                pk, sc_ = d["packed"][stor]
                T.pack_into(d["data"], g.L, g.S, stor, pk, sc_, stream=stream)
            batch.run(stream)
        e2e_step()
        stream.sync()
        ev0.record(stream)
        for _ in range(args.steps):
            e2e_step()
        ev1.record(stream)
        stream.sync()
        e2e_ms = ev0.elapsed_ms(ev1) / args.steps
        e2e = {"value": round(pairs / e2e_ms / 1e6, 2), "ms_per_step": round(e2e_ms, 3),
               "speedup_vs_plain_fp64": round(plain_ms / e2e_ms, 3),
               "includes": f"pack of the {len(dev)} cf32 bursts to {args.storage} "
                           f"(k_pack_scale + k_pack) + the batched kernel; cf32 inputs "
                           f"resident in HBM"}
        log(f"end to end (pack + batch): {e2e_ms:.2f} ms ({e2e['value']} GP/s)")
    else:
        e2e = {"value": round(mixed_gpps, 2), "ms_per_step": round(mixed_ms, 3),
               "speedup_vs_plain_fp64": round(plain_ms / mixed_ms, 3),
               "includes": "the batched kernel alone: cf32 samples are read as they are "
                           "(no pack); cf32 inputs resident in HBM"}

    # PCIe-inclusive (never the value): every step uploads the bursts' cf32
    # samples from pageable host memory through the library's pinned staging
    # chunks (tdbp_memcpy_htod_staged) on an upload stream, packs them there
    # for a packed storage, and runs them as batches of one subswath each on
    # the kernel stream, each waiting for its own uploads: the upload of one
    # subswath overlaps the batch of the one before.  Wall clock over 2 steps
    # after one warm-up.
    host = [d["data"].download() for d in dev]
    up = T.Stream()
    ngroup = max(1, min(nsub, len(dev)))
    per_group = -(-len(dev) // ngroup)
    groups = [list(range(i, min(len(dev), i + per_group)))
              for i in range(0, len(dev), per_group)]
    sub = []
    for gi in groups:
        b = T.Batch(T.MIXED, batch.variant)
        for i in gi:
            b.add(dev[i]["sc"].geom, smp(dev[i], stor), dev[i]["sat"], dev[i]["dem"],
                  dev[i]["out"])
        sub.append((gi, b, T.Event(), T.Event()))

    def h2d_step():
        for gi, b, ev, done in sub:
            up.wait(done)   # the previous step's batch of these bursts has read them
            for i in gi:
                dev[i]["data"].upload_staged(host[i], stream=up)
                if stor != T.CF32:
                    g = dev[i]["sc"].geom
                    pk, sc_ = dev[i]["packed"][stor]
                    T.pack_into(dev[i]["data"], g.L, g.S, stor, pk, sc_, stream=up)
            ev.record(up)
            stream.wait(ev)
            b.run(stream)
            done.record(stream)

    h2d_step()
    stream.sync()
    up.sync()
    t0 = time.perf_counter()
    for _ in range(2):
        h2d_step()
    stream.sync()
    up.sync()
    h2d_ms = (time.perf_counter() - t0) * 1e3 / 2
    h2d_bytes = sum(h.nbytes for h in host)
    del host
    e2e_h2d = {"value": round(pairs / h2d_ms / 1e6, 2), "ms_per_step": round(h2d_ms, 3),
               "upload_bytes": h2d_bytes,
               "includes": f"upload of the {len(dev)} bursts' cf32 samples from pageable host "
                           f"memory ({h2d_bytes / 1e9:.2f} GB) through pinned staging"
                           + ("" if stor == T.CF32 else f", pack to {args.storage}")
                           + f" + {len(sub)} batches of {per_group} bursts, each overlapping "
                             f"the next one's upload; wall clock"}
    log(f"end to end with the upload: {h2d_ms:.1f} ms ({e2e_h2d['value']} GP/s, "
        f"{h2d_bytes / h2d_ms / 1e6:.1f} GB/s of samples)")

    # The FP64 kernel batched the same way (one persistent launch).
    bp = T.Batch(T.PLAIN_FP64, -1)
    for d in dev:
        bp.add(d["sc"].geom, smp(d, T.CF32), d["sat"], d["dem"], d["out"])
    bp.run(stream)
    stream.sync()
    ev0.record(stream)
    for _ in range(args.plain_passes):
        bp.run(stream)
    ev1.record(stream)
    stream.sync()
    bplain_ms = ev0.elapsed_ms(ev1) / args.plain_passes
    bp.close()
    log(f"plain FP64 batched: {bplain_ms:.2f} ms ({pairs / bplain_ms / 1e6:.1f} GP/s)")

    # The other storage types, batched the same way (reported, not the value).
    others = {}
    for name, dt in dts.items():
        if dt == stor:
            continue
        b = make_batch(dt)
        b.run(stream)
        stream.sync()
        ev0.record(stream)
        for _ in range(max(3, args.steps // 4)):
            b.run(stream)
        ev1.record(stream)
        stream.sync()
        ms = ev0.elapsed_ms(ev1) / max(3, args.steps // 4)
        e_ph, e_amp = scene_error()
        others[name] = {"gpps": round(pairs / ms / 1e6, 1), "ms_per_step": round(ms, 3),
                        "phase_mrad_rms": round(e_ph * 1e3, 5), "amp_rel_rms": e_amp,
                        "meets_bar": bool(e_ph <= 1e-3 and e_amp <= 1e-4)}
        b.close()
        log(f"mixed {name}: {ms:.2f} ms ({pairs / ms / 1e6:.1f} GP/s), scene phase "
            f"{e_ph * 1e3:.4f} mrad amp {e_amp:.2e}")

    achieved = pairs * FLOP_PER_PAIR / (mixed_ms * 1e-3) / 1e12
    traffic, traffic_variant, busy = measured_traffic(args.storage, pairs, batch.variant)
    roof = {"bound": "valu", "achieved": round(achieved, 3), "peak": PEAK_FP32_TFLOPS,
            "unit": "TFLOP/s", "frac": round(achieved / PEAK_FP32_TFLOPS, 4),
            "traffic": traffic, "traffic_variant": traffic_variant,
            "unit_busy_pmc": busy,
            "kernel": "k_batch<MIXED> (persistent)", "flop_per_pair": FLOP_PER_PAIR,
            "pairs_per_launch": pairs,
            "plain_fp64_frac": round(pairs * FLOP_PER_PAIR / (plain_ms * 1e-3) / 1e12 /
                                     PEAK_FP64_TFLOPS, 4)}
    cpu = None
    if not args.no_cpu:
        cpu = cpu_baseline(dev[0]["sc"], dev[0]["data"])
        log(f"cpu baseline: {cpu}")

    line = {
        "metric": METRIC, "value": round(mixed_gpps, 2), "unit": "Gpixel·pulse/s",
        "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(mixed_ms, 3), "higher_is_better": True, "scaling": "weak",
        "vs_baseline": None, "dtype": "f32 (f64 per-tile reference)",
        "data": "synthetic (GPU-generated band-limited clutter + point targets, fBm DEM)",
        "config": {"workload": "IW scene: 3 subswaths x 9 uneven bursts (pulses U[1350,1550], "
                               "samples U[18000,25000], windows U[1000,4500] x U[1200,1600] "
                               "px), batched",
                   "bursts": len(dev), "pairs_per_step": pairs, "storage": args.storage,
                   "variant": batch.variant, "tile": T.variant_info(batch.variant)[:2]},
        "plain_fp64": {"value": round(plain_gpps, 2), "ms_per_pass": round(plain_ms, 3),
                       "launch": "one per burst",
                       "batched": {"value": round(pairs / bplain_ms / 1e6, 2),
                                   "ms_per_pass": round(bplain_ms, 3),
                                   "launch": "one persistent launch (k_batch_plain)"}},
        "speedup_vs_plain_fp64": round(plain_ms / mixed_ms, 3),
        "speedup_vs_plain_fp64_batched": round(bplain_ms / mixed_ms, 3),
        "end_to_end": e2e,
        "end_to_end_with_upload": e2e_h2d,
        "error_vs_fp64": {"phase_mrad_rms": round(ph * 1e3, 5), "amp_rel_rms": amp,
                          "meets_bar": bool(ph <= 1e-3 and amp <= 1e-4),
                          "against": "the FP64 kernel's images of the same bursts (the FP64 "
                                     "kernel is within 4.5e-8 rad / 1.4e-8 of the FP64 oracle "
                                     "on the 512-pulse burst), power-weighted over all "
                                     "computed pixels of the scene"},
        "other_storage": others,
        "roofline": roof,
        "cpu_baseline": cpu,
    }
    print(json.dumps(line), flush=True)
    batch.close()


if __name__ == "__main__":
    main()
