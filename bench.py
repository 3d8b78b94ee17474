#!/usr/bin/env python3
"""Benchmark driver: one JSON line with the headline measurement.

Headline (``value``): fused horizontal diffusion on a 512 x 512 x 160
float64 domain, halo 3, 64-byte aligned, layout (2, 1, 0), fields U[0,1)
from seed 0 - the plain-FP64 configuration the metric is quoted on.  A step
is one hdiff launch over the whole domain with the fields resident in HBM;
the caches (L2 and the 256 MB Infinity Cache) are flushed before every
timed launch, and each launch is timed with HIP events on the stream it
runs on.  ``value`` = compulsory bytes per launch / mean launch time.

Alongside, in the same process: GPU STREAM copy/scale/add/triad on three
2^29-element float64 arrays (the measured bandwidth ceiling), the 5-point
Laplacian on 512 x 512 x 160, vertical advection at 512 x 512 x 160 and
256 x 256 x 80 (float64, and float32 storage with float64 arithmetic), and
the OpenMP CPU baseline of hdiff on the same fields timed on this host.
"""

import argparse
import ctypes
import json
import os
import sys
import time
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

from stencil_benchmarks_amd import native  # noqa: E402
from stencil_benchmarks_amd.device import DeviceBuffer, DeviceField, geometry  # noqa: E402
from stencil_benchmarks_amd.tools import array  # noqa: E402

METRIC = "hdiff/vadv HBM GB/s & % of peak; batched-serve p50/p99 + speedup vs plain"
HBM_PEAK_GBS = 8000.0


def log(message):
    print(f"[bench] {message}", file=sys.stderr, flush=True)


def make_host_fields(domain, halo, dtype, count, seed, alignment=64):
    shape = tuple(d + 2 * h for d, h in zip(domain, halo))
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(count):
        a = array.alloc_array(shape, dtype, (2, 1, 0), alignment, halo)
        a[...] = rng.random(shape, dtype=np.float64).astype(dtype)
        out.append(a)
    return out


def device_fields_random(domain, halo, dtype, count, seed, alignment=64):
    """Device fields filled on the GPU (counter hash over the whole span)."""
    shape = tuple(d + 2 * h for d, h in zip(domain, halo))
    template = array.alloc_array(shape, dtype, (2, 1, 0), alignment, halo)
    fields = []
    code = native.SB_F64 if np.dtype(dtype) == np.float64 else native.SB_F32
    for f in range(count):
        dev = DeviceField(template, halo)
        n = dev.span // template.itemsize
        native.call("sb_stream_fill_random", code, ctypes.c_void_p(dev.base), n, seed * 16 + f)
        fields.append(dev)
    strides = [s // template.itemsize for s in template.strides]
    return fields, geometry(domain, strides, halo)


# Per-launch times come from events the dispatch records itself (hipExtLaunch-
# KernelGGL: the reference's 'hip-ext' timer).  Events recorded on the stream
# around the launch add about 2 us of marker latency per launch (measured on
# MI355X: hdiff 512x512x160 171.9 -> 169.5 us, vadv 256x256x80 float32
# storage 35.8 -> 33.7 us), which counts against the short kernels most.
TIMER = native.SB_TIMER_HIP_EXT


def time_launches(launch, steps, warmup, flush=True):
    """Warm up with `warmup` launches configured like the timed ones (cache
    flush included, so the flush buffer exists and the clocks have ramped),
    then time `steps` launches; returns per-launch seconds and wall."""
    for _ in range(warmup):
        seconds = ctypes.c_double(0.0)
        launch(native.launch_options(flush=flush, timer=TIMER), ctypes.byref(seconds))
    native.call("sb_synchronize")
    times = []
    start = time.perf_counter()
    for _ in range(steps):
        seconds = ctypes.c_double(0.0)
        launch(native.launch_options(flush=flush, timer=TIMER), ctypes.byref(seconds))
        times.append(seconds.value)
    native.call("sb_synchronize")
    wall = time.perf_counter() - start
    return np.array(times), wall


def hdiff_bytes(domain, itemsize):
    nx, ny, nz = domain
    return ((nx + 4) * (ny + 4) * nz + 2 * nx * ny * nz) * itemsize


def vadv_bytes(domain, itemsize):
    nx, ny, nz = domain
    return (5 * nx * ny * nz + (nx + 1) * ny * nz) * itemsize


def lap_bytes(domain, itemsize):
    nx, ny, nz = domain
    return ((nx + 2) * (ny + 2) * nz + nx * ny * nz) * itemsize


def bench_hdiff_headline(steps, warmup):
    domain, halo = (512, 512, 160), (3, 3, 3)
    host = make_host_fields(domain, halo, np.float64, 3, seed=0)
    host[2][...] = 0
    devs = [DeviceField(a, halo) for a in host]
    for d, a in zip(devs, host):
        d.upload(a)
    geom = geometry(domain, [s // 8 for s in host[0].strides], halo)
    ptrs = [ctypes.c_void_p(d.pointer()) for d in devs]

    def launch(opts, seconds):
        native.call("sb_hdiff", native.SB_F64, *ptrs, geom, opts, seconds)

    times, wall = time_launches(launch, steps, warmup)
    warm, _ = time_launches(launch, max(3, steps // 2), 0, flush=False)
    # the plugin boundary's round trip: host inp and coeff up, one launch,
    # out down (pageable numpy buffers, as the plugin mixin hands them over)
    native.call("sb_synchronize")
    start = time.perf_counter()
    devs[0].upload(host[0])
    devs[1].upload(host[1])
    launch(native.launch_options(), None)
    devs[2].download(host[2])
    native.call("sb_synchronize")
    round_trip = time.perf_counter() - start
    result = devs[2]
    gpu_out = np.ndarray(host[2].shape, np.float64,
                         buffer=np.zeros(result.span, np.uint8), strides=host[2].strides)
    result.download(gpu_out)
    return dict(domain=domain, halo=halo, host=host, gpu_out=gpu_out, times=times, wall=wall,
                warm_times=warm, bytes=hdiff_bytes(domain, 8), round_trip=round_trip,
                transfer_bytes=devs[0].span + devs[1].span + devs[2].span)


# launch shapes of the STREAM sweep (the reference sweeps block size x vector
# size, stream/cuda_hip.py:41-60, README.md:403-411): threads per block x
# elements per lane (float64: 1 or 2) x vectors per thread x non-temporal
# loads and stores x persistent grid (0: one pass, else workgroups per CU)
STREAM_SWEEP = [(block, vector, unroll, nt, per_cu)
                for block in (128, 256, 512, 1024)
                for vector in (1, 2)
                for unroll in (1, 2, 4)
                for nt in (0, 3)
                for per_cu in (0, 8)]


def bench_stream(repeats, shapes=None):
    """STREAM on three 2^29-element float64 arrays over the launch-shape
    sweep: per kernel the best bandwidth (GB/s) and the shape that gave it,
    each shape timed `repeats` times after one untimed launch."""
    n = 1 << 29
    bufs = [DeviceBuffer(n * 8) for _ in range(3)]
    for i, b in enumerate(bufs):
        native.call("sb_stream_fill_random", native.SB_F64, ctypes.c_void_p(b.ptr), n, 100 + i)
    words = {"copy": 2, "scale": 2, "add": 3, "triad": 3}
    best, shape_of, table = {}, {}, []
    for block, vector, unroll, nt, per_cu in shapes or STREAM_SWEEP:
        opts = native.launch_options(variant=nt, block=(block, vector, per_cu), unroll=unroll,
                                     timer=TIMER)
        for op, code in native.STREAM_OPS.items():
            times = []
            for _ in range(repeats + 1):
                seconds = ctypes.c_double(0.0)
                native.call("sb_stream_kernel", native.SB_F64, code,
                            *[ctypes.c_void_p(b.ptr) for b in bufs], n, 3.0, opts,
                            ctypes.byref(seconds))
                times.append(seconds.value)
            gbs = words[op] * n * 8 / min(times[1:]) / 1e9
            table.append((op, block, vector, unroll, nt, per_cu, gbs))
            if gbs > best.get(op, 0.0):
                best[op] = gbs
                shape_of[op] = {"block": block, "vector_elements": vector, "unroll": unroll,
                                "nontemporal": bool(nt), "workgroups_per_cu": per_cu}
    for b in bufs:
        b.free()
    return best, shape_of, table


def bench_lap(steps):
    domain, halo = (512, 512, 160), (3, 3, 3)
    devs, geom = device_fields_random(domain, halo, np.float64, 2, seed=3)
    ptrs = [ctypes.c_void_p(d.pointer()) for d in devs]

    def launch(opts, seconds):
        native.call("sb_laplacian", native.SB_F64, 1, 1, 0, *ptrs, geom, opts, seconds)

    times, _ = time_launches(launch, steps, 30)
    return lap_bytes(domain, 8) / times.mean() / 1e9, times.mean()


def bench_vadv(domain, dtype, precision, steps, variant=0):
    halo = (3, 3, 3)
    devs, geom = device_fields_random(domain, halo, dtype, 8, seed=4)
    ptr_array = (ctypes.c_void_p * 8)(*[d.pointer() for d in devs])

    def launch(opts, seconds):
        opts.variant = variant
        native.call("sb_vadv", precision, 0, ptr_array, geom, opts, seconds)

    times, _ = time_launches(launch, steps, 30)
    itemsize = np.dtype(dtype).itemsize
    return vadv_bytes(domain, itemsize) / times.mean() / 1e9, times.mean()


def bench_hdiff_f32(steps):
    domain, halo = (512, 512, 160), (3, 3, 3)
    devs, geom = device_fields_random(domain, halo, np.float32, 3, seed=5)
    ptrs = [ctypes.c_void_p(d.pointer()) for d in devs]

    def launch(opts, seconds):
        native.call("sb_hdiff", native.SB_F32_F64, *ptrs, geom, opts, seconds)

    times, _ = time_launches(launch, steps, 30)
    return hdiff_bytes(domain, 4) / times.mean() / 1e9, times.mean()


def bench_batched(compute_dtype, storage_dtype, repeats=2):
    """96 uneven subdomains x 10 steps of hdiff then vadv, one hipGraph, with
    launch shapes from the autotuner (tuned on scratch subdomains of the
    same shapes before the clock, or read from its cache)."""
    from stencil_benchmarks_amd import autotune, batch

    specs = batch.random_specs(96, 32, 512, 40, 160, seed=0)
    tuned = autotune.tune_batch(specs, storage_dtype, compute_dtype)
    subs = [batch.Subdomain(s.domain, s.halo, storage_dtype, seed=s.seed) for s in specs]
    plan = batch.Plan(subs, steps=10, compute=compute_dtype, hdiff_options=tuned.hdiff_options,
                      vadv_options=tuned.vadv_options)
    for _ in range(3):  # capture, then warm-up (the first launches on fresh fields run slower)
        plan.run(use_graph=True)
    native.call("sb_flush_caches")
    times = [plan.run(use_graph=True) for _ in range(repeats)]
    seconds = min(times)
    nbytes = 10 * sum(s.compulsory_bytes_per_step() for s in subs)
    points = 10 * sum(s.points for s in subs)
    plan.close()
    for s in subs:
        s.free()
    return {"seconds": seconds, "gbs": nbytes / seconds / 1e9,
            "gridpoint_steps_per_s": points / seconds, "subdomains": len(subs),
            "steps": 10, "points_per_step": points // 10,
            "autotuned": {"hdiff": tuned.hdiff, "vadv": tuned.vadv, "defaults": tuned.defaults,
                          "from_cache": tuned.from_cache, "candidates": len(tuned.trials)}}


def bench_plain_steps(steps=10, storage=np.float64, compute=np.float64):
    """The batched workload with the plain kernels: per subdomain and step one
    sb_hdiff and one sb_vadv launch, in the given storage and arithmetic
    types; kernel time only (sum of per-launch event times, so launch gaps do
    not count against the plain path)."""
    from stencil_benchmarks_amd import batch

    prec = native.precision_code(storage, compute)
    specs = batch.random_specs(96, 32, 512, 40, 160, seed=0)
    subs = [batch.Subdomain(s.domain, s.halo, storage, seed=s.seed) for s in specs]

    def one_step(sub, timed):
        """One hdiff + vadv step of `sub`; their kernel seconds when timed."""
        f = sub.fields
        cur, nxt = f[f"u{sub.parity}"], f[f"u{sub.parity ^ 1}"]
        seconds = [ctypes.c_double(0.0), ctypes.c_double(0.0)]
        refs = [ctypes.byref(x) if timed else None for x in seconds]
        native.call("sb_hdiff", prec, ctypes.c_void_p(cur.pointer()),
                    ctypes.c_void_p(f["coeff"].pointer()), ctypes.c_void_p(nxt.pointer()),
                    sub.geom, native.launch_options(timer=TIMER), refs[0])
        ptrs = [nxt, f["upos"], f["utens"], f["utensstage"], f["wcon"]]
        arr = (ctypes.c_void_p * 8)(*([p.pointer() for p in ptrs] + [0, 0, 0]))
        native.call("sb_vadv", prec, 0, arr, sub.geom, native.launch_options(timer=TIMER), refs[1])
        sub.advance(1)
        return seconds[0].value + seconds[1].value

    # untimed warm-up, as the batched runs get: two steps of every subdomain
    # (the first launches on fresh fields run slower)
    for sub in subs:
        for _ in range(2):
            one_step(sub, False)
    native.call("sb_synchronize")
    total = sum(one_step(sub, True) for sub in subs for _ in range(steps))
    nbytes = steps * sum(s.compulsory_bytes_per_step() for s in subs)
    for s in subs:
        s.free()
    return {"seconds": total, "gbs": nbytes / total / 1e9,
            "precision": f"{np.dtype(storage).name} storage, {np.dtype(compute).name} arithmetic"}


def bench_serving(count=160, load=0.8):
    """Poisson stream of hdiff+vadv requests, float32 storage, FP64 arithmetic."""
    from stencil_benchmarks_amd import serve

    from stencil_benchmarks_amd import autotune, batch

    mix = serve.poisson_requests(rate=0.0, count=count, seed=1)
    # launch shapes tuned on the mix's subdomain shapes (before the clock)
    tuned = autotune.tune_batch([batch.SubdomainSpec(r.domain) for r in mix], "float32", "float64")

    def server():
        return serve.Server(dtype="float32", compute="float64",
                            hdiff_options=tuned.hdiff_options, vadv_options=tuned.vadv_options)

    # warm-up: the same closed loop once untimed (the first launches on
    # fresh fields and a cold device run slower; with the tuning cached the
    # capacity run would otherwise be the first work of the leg)
    server().run(serve.poisson_requests(rate=0.0, count=count, seed=1), realtime=False)
    closed = server().run(mix, realtime=False)
    capacity = closed.requests / closed.wall_s
    rate = load * capacity
    stream = serve.poisson_requests(rate=rate, count=count, seed=1)
    served = server().run(stream, realtime=True)
    plain_s, plain_bytes, plain_points = serve.run_plain(
        serve.poisson_requests(rate=0.0, count=count, seed=1), dtype="float64")
    plain32_s, plain32_bytes, _ = serve.run_plain(
        serve.poisson_requests(rate=0.0, count=count, seed=1), dtype="float32",
        compute="float64")
    # open loop (Poisson arrivals at `load` x capacity): latencies; its
    # throughput is the arrival rate, so the speedup over plain FP64 is the
    # closed-loop (capacity) ratio on the same request mix
    out = served.summary()
    out.update({
        "rate_requests_per_s": rate,
        "load_fraction_of_capacity": load,
        "capacity_requests_per_s": capacity,
        "capacity_gbs": closed.bytes_moved / closed.wall_s / 1e9,
        "plain_f64_requests_per_s": count / plain_s,
        "plain_f64_gbs": plain_bytes / plain_s / 1e9,
        "plain_f32s_f64c_requests_per_s": count / plain32_s,
        "plain_f32s_f64c_gbs": plain32_bytes / plain32_s / 1e9,
        # continuous batching and float32 storage together (north-star ratio)
        "speedup_vs_plain_f64": capacity / (count / plain_s),
        # continuous batching alone: the same precision served one request at a time
        "speedup_vs_plain_same_precision": capacity / (count / plain32_s),
        "autotuned": {"hdiff": tuned.hdiff, "vadv": tuned.vadv, "defaults": tuned.defaults,
                      "from_cache": tuned.from_cache},
    })
    return out


def bench_host_stream(threads, array_size=1 << 27):
    """McCalpin STREAM on the host cores (3 x 1 GiB float64 arrays,
    non-temporal stores), GB/s per kernel: the memory ceiling of the CPU
    baseline, which runs on the same threads."""
    from stencil_benchmarks_amd.benchmarks_collection.stream import mc_calpin

    rows = mc_calpin.Native(array_size=array_size, ntimes=6, threads=threads).run()
    return {r["name"]: r["bandwidth"] / 1e3 for r in rows}


def host_threads():
    """Host threads for the CPU legs: OMP_NUM_THREADS when set, else every CPU
    this process may run on."""
    return int(os.environ.get("OMP_NUM_THREADS", "0")) or len(os.sched_getaffinity(0))


def host_description():
    """CPU model, the logical CPUs this process may run on and the physical
    cores among them (from /proc/cpuinfo), for the CPU legs' report."""
    allowed = os.sched_getaffinity(0)
    model, cores = "unknown", set()
    try:
        entry = {}
        for line in Path("/proc/cpuinfo").read_text().splitlines() + [""]:
            if not line.strip():
                if entry.get("processor") is not None and int(entry["processor"]) in allowed:
                    model = entry.get("model name", model)
                    cores.add((entry.get("physical id"), entry.get("core id")))
                entry = {}
                continue
            key, _, value = line.partition(":")
            entry[key.strip()] = value.strip()
    except (OSError, ValueError):
        pass
    return {"model": model, "logical_cpus": len(allowed), "physical_cores": len(cores) or None,
            "omp_proc_bind": os.environ.get("OMP_PROC_BIND"),
            "omp_places": os.environ.get("OMP_PLACES")}


def _time_cpu(call, budget_s, max_runs=5000):
    call()  # warm-up (first touch, thread spin-up)
    times, spent = [], 0.0
    while spent < budget_s and len(times) < max_runs:
        t = call()
        times.append(t)
        spent += t
    return float(np.median(times)), len(times), spent


def cpu_baseline(headline, budget_s=12.0):
    """OpenMP port of the reference CPU hdiff (Classic 8x8x1) on the headline
    fields: the `cpu_baseline` figure."""
    from oracle import oracle

    lib = oracle.cpu_lib()
    threads = host_threads()
    domain, halo = headline["domain"], headline["halo"]
    inp, coeff, out = headline["host"]
    strides = [s // 8 for s in inp.strides]

    def origin(a):
        return ctypes.c_void_p(a.ctypes.data + sum(s * h for s, h in zip(a.strides, halo)))

    args = [origin(inp), origin(coeff), origin(out)] + [ctypes.c_ssize_t(v) for v in (*domain, *strides)]
    best, runs, spent = _time_cpu(lambda: lib.cpu_hdiff_f64(*args, ctypes.c_int(threads)), budget_s)
    inner = tuple(slice(h, h + d) for d, h in zip(domain, halo))
    diff = float(np.abs(out[inner] - headline["gpu_out"][inner]).max())
    return {
        "value": headline["bytes"] / best / 1e9,
        "unit": "GB/s",
        "cores": threads,
        "kind": "port",
        "sample": f"hdiff 512x512x160 float64 full domain, OpenMP Classic 8x8x1 port, "
                  f"{runs} runs ({spent:.1f} s), median run",
        "seconds_per_pass": best,
        "max_abs_diff_vs_gpu": diff,
        "host": host_description(),
    }


def cpu_vadv_baseline(threads, budget_s=6.0):
    """OpenMP port of the reference CPU vadv (KMiddle, blocks of 8 columns)
    on a 512 x 512 x 160 float64 domain: GB/s of compulsory bytes."""
    from oracle import oracle

    lib = oracle.cpu_lib()
    domain, halo = (512, 512, 160), (3, 3, 3)
    fields = make_host_fields(domain, halo, np.float64, 5, seed=4)
    strides = [s // 8 for s in fields[0].strides]
    ptrs = [ctypes.c_void_p(a.ctypes.data + sum(s * h for s, h in zip(a.strides, halo)))
            for a in fields]
    args = ptrs + [ctypes.c_ssize_t(v) for v in (*domain, *strides)]
    best, runs, spent = _time_cpu(lambda: lib.cpu_vadv_f64(*args, ctypes.c_int(threads)),
                                  budget_s)
    return {"gbs": vadv_bytes(domain, 8) / best / 1e9, "seconds_per_pass": best,
            "cores": threads, "kind": "port",
            "sample": f"vadv 512x512x160 float64, OpenMP KMiddle port, {runs} runs "
                      f"({spent:.1f} s), median run"}


def numpy_config1(budget_s=5.0):
    """The reference's numpy OnTheFly hdiff at 128 x 128 x 80 (halo 3,
    float64, layout (0, 1, 2), inp and coeff U[0,1) from seed 0, out zero),
    timed by perf_counter around the numpy kernel like the reference's
    tools/timing.py; the reference formula's bytes over the median run."""
    from stencil_benchmarks_amd.benchmarks_collection.stencils.numpy import horizontal_diffusion

    bench = horizontal_diffusion.OnTheFly(domain=(128, 128, 80), halo=(3, 3, 3),
                                          dtype="float64", layout=(0, 1, 2), seed=0,
                                          verify=False)
    first = bench.run()  # verified once below, timed from the second run on
    times, spent = [], 0.0
    while spent < budget_s and len(times) < 200:
        result = bench.run()
        times.append(result["time"])
        spent += result["time"]
    checked = horizontal_diffusion.OnTheFly(domain=(128, 128, 80), halo=(3, 3, 3),
                                            dtype="float64", layout=(0, 1, 2), seed=0,
                                            verify=True)
    checked.run()
    best = float(np.median(times))
    return {"seconds": best, "reference_formula_gbs": bench.data_size / best / 1e9,
            "runs": len(times), "first_run_s": first["time"], "verified": True,
            "threads": 1, "note": "numpy elementwise kernels run on one thread"}


def sources_sha(paths):
    """sha256 over the named source files (relative to the repository)."""
    import hashlib

    digest = hashlib.sha256()
    for rel in paths:
        digest.update(rel.encode())
        digest.update((ROOT / rel).read_bytes())
    return digest.hexdigest()


def profiled_traffic(key):
    """HBM traffic per launch measured by rocprofv3 FETCH_SIZE/WRITE_SIZE runs
    (scaled by the copy-kernel calibration), committed in profiles/traffic.json;
    None unless the entry was measured on the kernel sources of this tree."""
    path = ROOT / "profiles" / "traffic.json"
    try:
        entry = json.loads(path.read_text())[key]
        if sources_sha(entry["sources"]) != entry["sources_sha256"]:
            log(f"profiles/traffic.json entry {key} was measured on other kernel sources")
            return None
        return entry["traffic_bytes"]
    except (OSError, KeyError, ValueError):
        return None


def main():
    parser = argparse.ArgumentParser()
    parser.add_argument("--gpus", type=int, default=1)
    parser.add_argument("--steps", type=int, default=20)
    # the first ~50 launches of a kernel on fresh fields run about 5 % slower
    # than the steady state (hdiff 512x512x160: 180.7 us, then 171.5 us;
    # busy-waiting the GPU beforehand does not remove it)
    parser.add_argument("--warmup", type=int, default=60)
    parser.add_argument("--quick", action="store_true", help="headline only")
    parser.add_argument("--only", choices=["hdiff", "hdiff_f32", "vadv", "laplacian", "stream",
                                           "stream_copy", "batched", "serving"],
                        help="run a single workload (profiling)")
    parser.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    args = parser.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only; --gpus {args.gpus} is not supported "
              "(the stencil path would shard by subdomain; one GPU runs one shard)",
              file=sys.stderr)
        sys.exit(2)

    native.init(0)
    info = native.device_info(0)
    log(f"device {info['name']} {info['arch']} CUs={info['compute_units']}")

    if args.only and args.only != "hdiff":
        run_single(args)
        return
    if args.only == "hdiff":
        args.quick = True
    log("hdiff 512x512x160 float64 (headline)")
    head = bench_hdiff_headline(args.steps, args.warmup)
    mean_s = float(head["times"].mean())
    achieved = head["bytes"] / mean_s / 1e9
    log(f"hdiff: {achieved:.1f} GB/s, mean launch {mean_s * 1e6:.1f} us")

    # the reference's own report for the same launches: bandwidth by its
    # data_size formula (2N + (nx+4)(ny+4)(nz+4)) * itemsize, and grid points/s
    nx, ny, nz = 512, 512, 160
    points = nx * ny * nz
    extras = {"hdiff_512x512x160_f64_pcie_inclusive": {
        "gbs": head["bytes"] / head["round_trip"] / 1e9, "seconds": head["round_trip"],
        "transfer_bytes": head["transfer_bytes"],
        "note": "host inp + coeff uploaded, one launch, out downloaded (pageable buffers)"},
        "hdiff_512x512x160_f64_reference_formula_gbs":
            (2 * points + (nx + 4) * (ny + 4) * (nz + 4)) * 8 / mean_s / 1e9,
        "hdiff_512x512x160_f64_gridpoints_per_s": points / mean_s}
    if not args.quick:
        log(f"STREAM 3 x 2^29 float64, {len(STREAM_SWEEP)} launch shapes")
        extras["stream_gbs"], extras["stream_best_shapes"], _ = bench_stream(3)
        extras["stream_shapes_swept"] = len(STREAM_SWEEP)
        log(f"STREAM best {extras['stream_gbs']}")
        log("laplacian 512x512x160 float64")
        extras["laplacian_gbs"], _ = bench_lap(args.steps)
        log("vadv")
        extras["vadv_512x512x160_f64_gbs"], vadv_s = bench_vadv((512, 512, 160), np.float64,
                                                                native.SB_F64, args.steps)
        # the reference's vadv data_size counts ccol/dcol traffic: 10 N * itemsize
        extras["vadv_512x512x160_f64_reference_formula_gbs"] = 10 * points * 8 / vadv_s / 1e9
        extras["vadv_512x512x160_f64_gridpoints_per_s"] = points / vadv_s
        extras["vadv_256x256x80_f64_gbs"], _ = bench_vadv((256, 256, 80), np.float64,
                                                          native.SB_F64, args.steps)
        extras["vadv_256x256x80_f32s_f64c_gbs"], _ = bench_vadv((256, 256, 80), np.float32,
                                                                native.SB_F32_F64, args.steps)
        extras["vadv_512x512x160_f32s_f64c_gbs"], _ = bench_vadv((512, 512, 160), np.float32,
                                                                 native.SB_F32_F64, args.steps)
        extras["hdiff_512x512x160_f32s_f64c_gbs"], _ = bench_hdiff_f32(args.steps)
        extras["hdiff_512x512x160_f64_warm_gbs"] = head["bytes"] / float(head["warm_times"].mean()) / 1e9

        triad = extras["stream_gbs"]["triad"]
        extras["hdiff_frac_of_triad"] = achieved / triad
        extras["vadv_512x512x160_f64_frac_of_triad"] = extras["vadv_512x512x160_f64_gbs"] / triad
        extras["vadv_256x256x80_f64_frac_of_triad"] = extras["vadv_256x256x80_f64_gbs"] / triad
        log("batched: 96 subdomains x 10 steps (float64, float32 storage)")
        b64 = bench_batched(np.float64, np.float64)
        b32 = bench_batched(np.float64, np.float32)
        extras["batched_f64"] = b64
        extras["batched_f32s_f64c"] = b32
        extras["batched_f32_speedup_vs_f64"] = b64["seconds"] / b32["seconds"]
        plain = bench_plain_steps()
        plain32 = bench_plain_steps(storage=np.float32, compute=np.float64)
        extras["plain_f64_same_workload"] = plain
        extras["plain_f32s_f64c_same_workload"] = plain32
        # batching alone: batched vs plain kernels in the same precision
        extras["batched_speedup_vs_plain_same_precision"] = {
            "f64": plain["seconds"] / b64["seconds"],
            "f32s_f64c": plain32["seconds"] / b32["seconds"]}
        # batching and float32 storage together (the north-star ratio): the
        # float32-storage batch against the plain FP64 kernels
        extras["batched_f32_speedup_vs_plain_f64"] = plain["seconds"] / b32["seconds"]
        log(f"batched f64 {b64['gbs']:.0f} GB/s, f32 {b32['gbs']:.0f} GB/s, plain f64 "
            f"{plain['gbs']:.0f} GB/s, plain f32 {plain32['gbs']:.0f} GB/s: f32 batched "
            f"{extras['batched_f32_speedup_vs_plain_f64']:.2f}x plain f64")
        log("serving: Poisson stream at 80% of capacity")
        extras["serving"] = bench_serving()
        log(f"serving p50 {extras['serving']['p50_latency_ms']:.2f} ms "
            f"p99 {extras['serving']['p99_latency_ms']:.2f} ms, "
            f"speedup vs plain f64 {extras['serving']['speedup_vs_plain_f64']:.2f}")

    baseline = None
    if not args.no_cpu:
        log("CPU baseline (OpenMP port) on the headline fields")
        baseline = cpu_baseline(head)
        log("CPU baseline: vadv KMiddle port")
        baseline["vadv_512x512x160_f64"] = cpu_vadv_baseline(baseline["cores"])
        log("CPU baseline: numpy OnTheFly hdiff 128x128x80 (the reference's CPU case)")
        baseline["numpy_hdiff_128x128x80_f64"] = numpy_config1()
        log("host STREAM (the CPU baseline's memory ceiling)")
        baseline["host_stream_gbs"] = bench_host_stream(baseline["cores"])
        baseline["frac_of_host_triad"] = baseline["value"] / baseline["host_stream_gbs"]["triad"]

    record = {
        "metric": METRIC,
        "value": achieved,
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": head["wall"] / args.steps * 1e3,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic: fields uniform[0,1) from seed 0, resident in HBM, caches flushed "
                "before each timed launch",
        "config": {
            "workload": "hdiff 512x512x160 halo 3 float64, 64-byte aligned, layout (2,1,0)",
            "domain": [512, 512, 160],
            "halo": [3, 3, 3],
            "kernel": "sb_hdiff default: variant 2 (64x8 LDS tile staged by global-to-LDS loads)",
            "compulsory_bytes_per_launch": head["bytes"],
            "device": info["name"] or f"{info['arch']} ({info['compute_units']} CUs)",
        },
        "roofline": {
            "bound": "hbm",
            "achieved": achieved,
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": achieved / HBM_PEAK_GBS,
            "traffic": profiled_traffic("hdiff_512x512x160_f64"),
        },
        "cpu_baseline": baseline,
        "kernel_mean_us": mean_s * 1e6,
        "extras": extras,
    }
    print(json.dumps(record))


def run_single(args):
    """One workload only, printed as JSON (used under rocprofv3)."""
    out = {"workload": args.only}
    if args.only == "vadv":
        out["vadv_512x512x160_f64_gbs"], out["mean_s"] = bench_vadv(
            (512, 512, 160), np.float64, native.SB_F64, args.steps)
        out["vadv_512x512x160_f32s_f64c_gbs"], out["mean_s_f32s"] = bench_vadv(
            (512, 512, 160), np.float32, native.SB_F32_F64, args.steps)
        out["vadv_256x256x80_f64_gbs"], out["mean_s_256"] = bench_vadv(
            (256, 256, 80), np.float64, native.SB_F64, args.steps)
        out["vadv_256x256x80_f32s_f64c_gbs"], out["mean_s_256_f32s"] = bench_vadv(
            (256, 256, 80), np.float32, native.SB_F32_F64, args.steps)
    elif args.only == "hdiff_f32":
        out["hdiff_512x512x160_f32s_f64c_gbs"], out["mean_s"] = bench_hdiff_f32(args.steps)
    elif args.only == "laplacian":
        out["laplacian_gbs"], out["mean_s"] = bench_lap(args.steps)
    elif args.only == "stream":
        out["stream_gbs"], out["stream_best_shapes"], table = bench_stream(3)
        out["stream_sweep"] = table
    elif args.only == "stream_copy":
        # one plain shape (counter calibration: bytes read and written are known)
        out["stream_gbs"], out["stream_best_shapes"], _ = bench_stream(3, [(256, 2, 1, 0, 0)])
    elif args.only == "batched":
        out["batched_f64"] = bench_batched(np.float64, np.float64)
        out["batched_f32s_f64c"] = bench_batched(np.float64, np.float32)
    elif args.only == "serving":
        out["serving"] = bench_serving(count=60)
    print(json.dumps(out))


if __name__ == "__main__":
    main()
