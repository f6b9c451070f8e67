"""Benchmark: batched transforms/s and HBM roofline fraction of the MI355X 3D FFT.

One step = one forward execute of the headline workload (17x17x17 complex128, batch 1024,
inputs iid uniform(-1,1)) on device-resident buffers.  Each step uses the next of R
(in, out) buffer pairs, R chosen so the pairs total >= 2 GiB: every working set here fits
the MI355X's 256 MB Infinity Cache, so same-buffer repetition would time the cache, not
HBM.  After W warm-up steps, exactly K steps are timed between HIP events on the launch
stream, bracketed by device synchronisations (the contract region); then 5 windows of n
steps each, n calibrated so a window lasts >= 20 ms, run back to back, and the reported
rate (value, ms_per_step, roofline) is the median window's, with the spread of the windows
under "timing" (short regions catch the clock ramp: the reference's driver insists on
>= 20 ms samples for the same reason).  The other workloads (8^3 x 4096, 36^3 x 128,
24x24x48 x 64, the 17^3 inverse, and 24^3 x 512, the largest batch of the serving mix's
24^3 requests) are timed the same way and reported under "secondary".

"precision_variants": complex64 on the uneven batch set 6^3 x 65536, 8^3 x 32768,
12^3 x 8192, 17^3 x 2048 -- as one persistent mixed launch (FFT, and the DFT-as-matrix
matrix-core form), as per-geometry FFT plans, and as per-geometry matrix-core plans (split
bf16 / fp16, three products, FP32 accumulate) -- with relative L2 and max error on 256
volumes per geometry against
numpy.fft in float64, and for the matrix-core kernels the executed MFMA TFLOP/s against the
2.5 PFLOP/s dense peak.

"small_batch_latency": batch-1 complex128 executes of every cube geometry, device time back
to back and host round trip, launched directly and replayed from a captured graph.

"host_abi": the reference's host-pointer ABI (fft3d_create / fft3d_execute) at 17^3 x 1024:
copies in and out of pageable host memory inside every execute (through pinned staging, in
pipelined chunks), so the rate is the host side's and the host link's, reported beside the
device-resident value, never as it.

"serving": the request server under Poisson arrivals (20,000 requests, the mixed stream of
opt-fft_amd/serving.py, 64 GB budget, 16 streams, 30 us batching window for the
continuously batched server): the highest arrival rate whose p99 latency stays
within 2 ms, for continuous batching and for the two plain one-launch-per-request paths
(synchronous, and asynchronous with 16 launches in flight on the same streams), the
throughput ratio of batching to each at that cap, and each mode's results checked on a
sampled burst against numpy.fft.

Prints ONE JSON line: the contract's fields and of the rest the figures (BRIEF), under 7,000 bytes,
so that whoever keeps only the end of the output has the whole of it.  --record PATH writes the
full record, every load point, window and candidate, as JSON.  `python bench.py --gpus N` with N > 1 exits: the benchmark runs on one
GPU (batches of independent volumes shard by volume with no communication).
"""
import argparse
import json
import math
import os
import re
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_HBM_GBS = 8000.0
# HBM bytes per launch of the headline kernel (pipe_17x17x17_c128_fwd_v2t640p1_fold_st3, the
# race's pick) from rocprofv3 FETCH_SIZE + WRITE_SIZE, each scaled by the same counter on the
# runtime's copy of a known size: 39,988.7 KiB x 2 + 78,978.4 KiB
# (profiles/k_fpipe_17x17x17_c128_fwd_b1024.md).
TRAFFIC = int((39988.65625 * 2 + 78978.421875) * 1024)
TRAFFIC_KERNEL = "pipe_17x17x17_c128_fwd_v2t640p1_fold_st3"
ROTATE_BYTES = 2 << 30

HEADLINE = dict(name="L17_c128_fwd_b1024", shape=(17, 17, 17), batch=1024, dist="uniform",
                direction=-1)
SECONDARY = [
    dict(name="L8_c128_fwd_b4096", shape=(8, 8, 8), batch=4096, dist="uniform", direction=-1),
    dict(name="L17_c128_bwd_b1024", shape=(17, 17, 17), batch=1024, dist="uniform",
         direction=+1),
    dict(name="L36_c128_fwd_b128", shape=(36, 36, 36), batch=128, dist="normal_half",
         direction=-1),
    dict(name="24x24x48_c128_fwd_b64", shape=(24, 24, 48), batch=64, dist="normal_half",
         direction=-1),
    dict(name="L24_c128_fwd_b512", shape=(24, 24, 24), batch=512, dist="uniform",
         direction=-1),
]


def make_input(shape, batch, seed, dist):
    rng = np.random.default_rng(seed)
    full = (batch,) + tuple(shape)
    if dist == "uniform":
        re, im = rng.uniform(-1, 1, full), rng.uniform(-1, 1, full)
    else:
        s = math.sqrt(0.5)
        re, im = rng.normal(0, s, full), rng.normal(0, s, full)
    return (re + 1j * im).astype(np.complex128)


# Accuracy of a measured output, against numpy.fft in float64 (the reference's boundary check,
# bench/geom/check.py:28-33); the unnormalised backward transform is V * ifftn.
def _np_dft(x, sign=-1):
    x = np.asarray(x, dtype=np.complex128)
    if sign < 0:
        return np.fft.fftn(x, axes=(-3, -2, -1))
    return np.fft.ifftn(x, axes=(-3, -2, -1)) * (x.shape[-3] * x.shape[-2] * x.shape[-1])


def _rel_l2(y, ref):
    return float(np.linalg.norm((np.asarray(y, np.complex128) - ref).ravel()) /
                 np.linalg.norm(ref.ravel()))


def _rel_max(y, ref):
    return float(np.max(np.abs(np.asarray(y, np.complex128) - ref)) / np.max(np.abs(ref)))


def measure(pkg, wl, steps, warmup, check=True, windows=5, window_ms=20.0):
    """Time one workload.  After `warmup` untimed executes: (1) exactly `steps` executes
    between HIP events on the launch stream, bracketed by device synchronisations (the
    contract region); (2) `windows` back-to-back windows of n executes each, n calibrated
    from (1) so that a window lasts >= window_ms (the >= 20 ms samples of the reference's
    driver, bench/gpu/driver.cu:17-32: shorter samples catch the clock ramp).  The windows
    follow each other on the stream with no synchronisation between them, so the device
    stays busy through all of them.  The reported rate is the median window's."""
    f, h = pkg.fft3d, pkg.hip
    shape, batch = wl["shape"], wl["batch"]
    V = shape[0] * shape[1] * shape[2]
    nbytes = V * batch * 16
    rot = max(1, math.ceil(ROTATE_BYTES / (2 * nbytes)))
    x = make_input(shape, batch, seed=2024 + batch, dist=wl["dist"])
    ins = [h.DeviceBuffer(nbytes) for _ in range(rot)]
    outs = [h.DeviceBuffer(nbytes) for _ in range(rot)]
    ins[0].upload(x)
    for b in ins[1:]:
        h.check(h.lib().hipMemcpy(b.ptr, ins[0].ptr, nbytes, h.D2D), "hipMemcpy D2D")
    plan = f.Plan(shape, batch, wl["direction"], f.C128)
    stream = h.Stream()
    e0, e1 = h.Event(), h.Event()
    k = 0

    def step():
        nonlocal k
        plan.execute(ins[k % rot].addr, outs[k % rot].addr, stream=stream)
        k += 1

    for _ in range(warmup):
        step()
    h.synchronize()
    e0.record(stream)
    for _ in range(steps):
        step()
    e1.record(stream)
    e1.synchronize()
    h.synchronize()
    contract_ms = e0.elapsed_ms(e1)
    # 25% margin: the contract region includes the clock ramp and runs slower
    n = max(steps, math.ceil(1.25 * window_ms / (contract_ms / steps)))
    evs = [h.Event() for _ in range(windows + 1)]
    evs[0].record(stream)
    for w in range(windows):
        for _ in range(n):
            step()
        evs[w + 1].record(stream)
    evs[-1].synchronize()
    h.synchronize()
    last_out = (k - 1) % rot
    wms = sorted(evs[w].elapsed_ms(evs[w + 1]) for w in range(windows))
    for e in evs:
        e.close()
    med = wms[windows // 2] / n
    res = dict(kernel=plan.kernel, rotate_pairs=rot, steps=steps,
               contract_ms_total=contract_ms, contract_ms_per_execute=contract_ms / steps,
               windows=windows, executes_per_window=n,
               window_ms=[round(v, 4) for v in wms],
               window_spread=(wms[-1] - wms[0]) / wms[windows // 2],
               ms_per_execute=med, transforms_per_s=batch / (med * 1e-3),
               us_per_execute_min=wms[0] / n * 1e3, us_per_execute_max=wms[-1] / n * 1e3)
    # Kernel duration for the roofline: the median window's time per execute (one kernel per
    # execute for the fused paths; the whole two-kernel sequence for pencils).
    algo = 2.0 * nbytes
    res["algorithmic_bytes_per_execute"] = algo
    res["achieved_GBs"] = algo / (med * 1e-3) / 1e9
    res["roofline_frac"] = res["achieved_GBs"] / PEAK_HBM_GBS
    if check:
        # every input buffer holds x
        y = outs[last_out].download(np.complex128, x.shape)
        res["rel_l2_vs_numpy"] = _rel_l2(y, _np_dft(x, wl["direction"]))
    for b in ins + outs:
        b.close()
    stream.close()
    plan.close()
    return res


# The reference's CPU kernels, each linked with the reference's own timing driver
# (bench/geom/driver.c single-core, bench/mt/driver.c OpenMP; built into oracle/_ref by
# oracle/build_ref.sh), timed at the GPU configurations' batches.  Per geometry: the
# single-core best-exemplar candidates (winner and alternate of bench/geom/best/fft3d_best.c's
# table) and the multi-threaded round's kernels; the faster candidate is reported, as the
# reference's race-at-create picks it.
CPU_CASES = [(17, 1024, "uniform"), (8, 4096, "uniform"), (36, 128, "normal_half"),
             (6, 65536, "uniform")]
CPU_ST = {6: ["L6_pfa", "L6_unrolled"], 8: ["L8_batchsimd", "L8_fusedaxes"],
          17: ["L17_matrixsimd", "L17_rader"], 36: ["L36_mixedradix", "L36_pfa", "L36_pencilfused"]}
CPU_MT = {6: ["L6_pfa"], 8: ["L8_fusedaxes", "L8_batchsimd"], 17: ["L17_winograd", "L17_matrixsimd"],
          36: ["L36_mixedradix", "L36_pfa"]}


def _ref_dir():
    isa = "v4" if "avx512f" in open("/proc/cpuinfo").read() else "v3"
    d = os.path.join(ROOT, "oracle", "_ref", isa)
    return d if os.path.isdir(d) else None


def _ref_driver(exe, L, batch, fin, env, pin=None, samples=10):
    """One run of the reference driver: warm-up, inner count calibrated to >= 20 ms samples,
    `samples` timed samples (bench/geom/driver.c:166-189).  Returns its JSON record."""
    import subprocess
    import tempfile
    with tempfile.NamedTemporaryFile(suffix=".json") as js:
        cmd = ([] if pin is None else ["taskset", "-c", str(pin)]) + [
            exe, "--L", str(L), "--batch", str(batch), "--in", fin, "--json", js.name,
            "--samples", str(samples), "--warmup", "2", "--min-sample-ms", "20"]
        r = subprocess.run(cmd, capture_output=True, text=True, env=env, timeout=300)
        if r.returncode != 0:
            return None
        return json.loads(open(js.name).read())


def cpu_baseline():
    """The reference's own CPU path on this host's cores through its own driver (kind
    "reference"): all cores (OpenMP, OMP_NUM_THREADS = the cores this process may use,
    PROC_BIND=close, PLACES=cores) and one pinned core, for every geometry of the GPU
    configurations at their batches (6^3 at 65536 in complex128, the CPU path's only
    precision).  value = the headline's (17^3 x 1024) all-core rate from the driver's
    fastest sample.  Falls back to timing the oracle's numpy.fft ("port")."""
    import tempfile
    d = _ref_dir()
    if d:
        cores = sorted(os.sched_getaffinity(0))
        env = dict(os.environ, OMP_NUM_THREADS=str(len(cores)), OMP_PROC_BIND="close",
                   OMP_PLACES="cores")
        model = ""
        try:
            model = [l.split(":", 1)[1].strip() for l in open("/proc/cpuinfo")
                     if l.startswith("model name")][0]
        except Exception:
            pass
        per = {}
        with tempfile.TemporaryDirectory() as tmp:
            for L, batch, dist in CPU_CASES:
                fin = os.path.join(tmp, f"in{L}.bin")
                make_input((L, L, L), batch, seed=2024 + batch, dist=dist).tofile(fin)
                row = {"batch": batch}
                for kind, table, pin, e in (("single_core", CPU_ST, cores[0], None),
                                            ("all_cores", CPU_MT, None, env)):
                    cands = []
                    for k in table[L]:
                        exe = os.path.join(d, "st" if pin is not None else "mt", k)
                        rec = _ref_driver(exe, L, batch, fin, e, pin) if os.path.exists(exe) else None
                        if rec:
                            pe = rec["per_execute_seconds"]
                            cands.append(dict(kernel=k, value=batch / pe["min"],
                                              value_median=batch / pe["median"],
                                              inner=rec["inner"], samples=rec["samples"]))
                    if cands:
                        best = max(cands, key=lambda c: c["value"])
                        row[kind] = dict(best, cores=1 if pin is not None else len(cores),
                                         candidates=cands)
                os.remove(fin)
                per[f"L{L}"] = row
                print(f"# cpu_baseline L={L}: {row}", file=sys.stderr, flush=True)
        head = per.get("L17", {}).get("all_cores")
        if head:
            return dict(value=head["value"], unit="transforms/s", cores=head["cores"],
                        kind="reference",
                        sample=f"reference {head['kernel']} (bench/mt/impl_4, OpenMP, "
                               f"{head['cores']} threads) through the reference's driver "
                               f"(bench/mt/driver.c: >=20 ms samples, fastest of "
                               f"{head['samples']}) on 17^3 complex128 x 1024 on {model}; "
                               f"FFTW not built (needs its configure-generated config.h)",
                        single_core=per["L17"].get("single_core"),
                        per_geometry=per)
    import oracle
    x = make_input((17, 17, 17), 64, seed=7, dist="uniform")
    n, t0 = 0, time.perf_counter()
    while time.perf_counter() - t0 < 10.0:
        oracle.fftn_numpy(x)
        n += x.shape[0]
    dt = time.perf_counter() - t0
    return dict(value=n / dt, unit="transforms/s", cores=1, kind="port",
                sample=f"numpy.fft.fftn (pocketfft) on 64 x 17^3 complex128 volumes, "
                       f"repeated for {dt:.1f} s ({n} transforms), 1 thread")


# Precision variants on uneven batches (complex64): one persistent mixed launch, the
# per-geometry complex64 FFT plans, and the DFT-as-matrix variant on the matrix cores.
UNEVEN_MIX = [((6, 6, 6), 65536), ((8, 8, 8), 32768), ((12, 12, 12), 8192), ((17, 17, 17), 2048)]
MIX_CHECK = 256          # volumes per item compared with numpy.fft in float64
PEAK_MFMA_TFLOPS = 2500.0   # dense bf16/fp16 matrix peak of one MI355X


def _uniform_c64(rng, shape, batch):
    full = (batch,) + tuple(shape)
    return (rng.uniform(-1, 1, full) + 1j * rng.uniform(-1, 1, full)).astype(np.complex64)


# Volumes per block of the mixed matrix-core launch; a standalone kernel's is in its name
# ("_v<VPW>t").
MFMA_VPW = {(6, 6, 6): 16, (8, 8, 8): 8, (12, 12, 12): 2, (17, 17, 17): 1, (8, 8, 16): 4}


def mfma_flops(shape, nvol, kernel=""):
    """MFMA flops the matrix-core kernel executes for nvol volumes: per block of VPW volumes
    and per axis pass of length N, ceil(lines/16) tiles of TM x TK x 3 products (three per
    tile for the compensated split), TM = ceil(2N/16); K = 16 instructions (TK = ceil(2N/16),
    2*16*16*16 flops each), or K = 32 ones (TK = ceil(2N/32), 2*16*16*32 flops each) on the
    axes with 2N > 16 of a "k32" kernel and of the mixed launch; the 17-point tiles of a
    "fold" kernel and of the mixed launch are 2 x 3 K = 32 products."""
    m = re.search(r"_v(\d+)t\d+", kernel)
    vpw = int(m.group(1)) if m else MFMA_VPW[tuple(shape)]
    V = shape[0] * shape[1] * shape[2]

    def per(nv):
        fl = 0.0
        for n in shape:
            if n == 17 and ("fold" in kernel or kernel.startswith("multi_")):   # 2 x 3 K = 32
                fl += -(-(nv * V // n) // 16) * 2 * 3 * 2.0 * 16 * 16 * 32
                continue
            kw = 32 if (2 * n > 16 and ("k32" in kernel or kernel.startswith("multi_"))) else 16
            tm, tk = (2 * n + 15) // 16, (2 * n + kw - 1) // kw
            fl += -(-(nv * V // n) // 16) * tm * tk * 3 * 2.0 * 16 * 16 * kw
        return fl
    full, part = divmod(nvol, vpw)
    return full * per(vpw) + (per(part) if part else 0.0)


def precision_mix(pkg, steps=20):
    f, h = pkg.fft3d, pkg.hip
    rng = np.random.default_rng(44)
    xs = [_uniform_c64(rng, sh, b) for sh, b in UNEVEN_MIX]
    nbytes = sum(x.nbytes for x in xs)
    # Input/output sets rotated so that >= 2 GiB pass between two uses of one set: the
    # mix (882 MB in + out) and each item alone would otherwise stay in the 256 MB
    # Infinity Cache between launches.
    sets = max(3, math.ceil(ROTATE_BYTES / (2 * nbytes)) + 1)
    ins = [[h.DeviceBuffer(x.nbytes) for x in xs] for _ in range(sets)]
    outs = [[h.DeviceBuffer(x.nbytes) for x in xs] for _ in range(sets)]
    for s_ in range(sets):
        for b, x in zip(ins[s_], xs):
            b.upload(x)
    stream = h.Stream()
    e0, e1 = h.Event(), h.Event()

    def timed(launch, nrot):
        """Seconds per launch: the median of 3 back-to-back windows of >= 20 ms, the launch
        argument cycling through nrot buffer sets."""
        i = 0
        for _ in range(3):
            launch(i % nrot)
            i += 1
        h.synchronize()
        e0.record(stream)
        for _ in range(5):
            launch(i % nrot)
            i += 1
        e1.record(stream)
        e1.synchronize()
        n = max(steps, math.ceil(25.0 / (e0.elapsed_ms(e1) / 5)))
        evs = [h.Event() for _ in range(4)]
        evs[0].record(stream)
        for w in range(3):
            for _ in range(n):
                launch(i % nrot)
                i += 1
            evs[w + 1].record(stream)
        evs[-1].synchronize()
        ws = sorted(evs[w].elapsed_ms(evs[w + 1]) for w in range(3))
        for e in evs:
            e.close()
        return ws[1] / n * 1e-3

    def errors(bufs):
        out = {}
        for (sh, b), x, ob in zip(UNEVEN_MIX, xs, bufs):
            y = ob.download(np.complex64, x.shape)[:MIX_CHECK]
            ref = _np_dft(x[:MIX_CHECK])
            out[f"L{sh[0]}"] = dict(rel_l2=_rel_l2(y, ref), rel_max=_rel_max(y, ref))
        return out

    res = {"items": [dict(shape=list(sh), batch=b) for sh, b in UNEVEN_MIX],
           "bytes_per_launch": 2 * nbytes, "error_sample_volumes": MIX_CHECK}
    mp = f.MultiPlan([(sh, b, -1) for sh, b in UNEVEN_MIX], f.C64)
    t = timed(lambda s_: mp.execute([b.addr for b in ins[s_]], [b.addr for b in outs[s_]],
                                    stream=stream), sets)
    h.synchronize()
    res["one_launch_fft_c64"] = dict(kernel=mp.info()[0], us=t * 1e6, GBs=2 * nbytes / t / 1e9,
                                     errors=errors(outs[0]))
    mp.close()
    for tag, flag in (("one_launch_mfma_bf16x3", f.MFMA_BF16), ("one_launch_mfma_fp16x3", f.MFMA_FP16)):
        mp = f.MultiPlan([(sh, b, -1) for sh, b in UNEVEN_MIX], f.C64, flags=flag)
        t = timed(lambda s_: mp.execute([b.addr for b in ins[s_]], [b.addr for b in outs[s_]],
                                        stream=stream), sets)
        h.synchronize()
        fl = sum(mfma_flops(sh, b, mp.info()[0]) for sh, b in UNEVEN_MIX)
        res[tag] = dict(kernel=mp.info()[0], us=t * 1e6, GBs=2 * nbytes / t / 1e9,
                        mfma_tflops=fl / t / 1e12, mfma_util=fl / t / 1e12 / PEAK_MFMA_TFLOPS,
                        errors=errors(outs[0]))
        mp.close()
    for lst in ins + outs:
        for b in lst:
            b.close()
    # Per-geometry plans: each item with its own rotation of >= 2 GiB.
    for tag in ("fft_c64", "mfma_bf16x3", "mfma_fp16x3"):
        res[tag] = {}
    for (sh, b), x in zip(UNEVEN_MIX, xs):
        nrot = math.ceil(ROTATE_BYTES / (2 * x.nbytes)) + 1
        bi = [h.DeviceBuffer(x.nbytes) for _ in range(nrot)]
        bo = [h.DeviceBuffer(x.nbytes) for _ in range(nrot)]
        bi[0].upload(x)
        for q in bi[1:]:
            h.check(h.lib().hipMemcpy(q.ptr, bi[0].ptr, x.nbytes, h.D2D), "hipMemcpy D2D")
        ref = _np_dft(x[:MIX_CHECK])
        for tag, flag in (("fft_c64", 0), ("mfma_bf16x3", f.MFMA_BF16),
                          ("mfma_fp16x3", f.MFMA_FP16)):
            p = f.Plan(sh, b, f.FORWARD, f.C64, flags=flag)
            tk = timed(lambda s_: p.execute(bi[s_].addr, bo[s_].addr, stream=stream), nrot)
            h.synchronize()
            d = dict(kernel=p.kernel, us=tk * 1e6, GBs=2 * x.nbytes / tk / 1e9, rotate_sets=nrot)
            y = bo[0].download(np.complex64, x.shape)[:MIX_CHECK]
            d["rel_l2"] = _rel_l2(y, ref)
            d["rel_max"] = _rel_max(y, ref)
            if flag:
                fl = mfma_flops(sh, b, p.kernel)
                d["mfma_tflops"] = fl / tk / 1e12
                d["mfma_util"] = d["mfma_tflops"] / PEAK_MFMA_TFLOPS
            res[tag][f"L{sh[0]}"] = d
            p.close()
        for q in bi + bo:
            q.close()
    res["rotate_sets_mix"] = sets
    return res


def _serving_check(pkg, srv, pools, n=300, seed=21):
    """Sampled results of one burst of the request mix through `srv`, outputs in caller
    buffers: the first and last volume of every request against numpy.fft in float64.
    Returns the worst relative L2 per precision."""
    import ctypes
    f, h, sv = pkg.fft3d, pkg.hip, pkg.serving
    mix = sv.draw_mix(n, seed=seed)
    rng = np.random.default_rng(seed)
    firsts = [int(rng.integers(0, sv.MAX_BATCH + 1)) for _ in mix]
    sizes = [b * s_[0] * s_[1] * s_[2] * (16 if p == f.C128 else 8) for s_, b, _, p in mix]
    offs = np.concatenate([[0], np.cumsum([(z + 255) // 256 * 256 for z in sizes])])
    arena = h.DeviceBuffer(int(offs[-1]))
    reqs = [f.SrvRequest(*s_, b, d, p, pools.addr(s_, p, first), arena.addr + int(o))
            for (s_, b, d, p), first, o in zip(mix, firsts, offs[:-1])]
    srv.run_trace(reqs, np.linspace(0.0, 2e-3, n))
    worst = {"c128": 0.0, "c64": 0.0}
    for (s_, b, d, p), first, o in zip(mix, firsts, offs[:-1]):
        V = s_[0] * s_[1] * s_[2]
        dt = np.complex128 if p == f.C128 else np.complex64
        for i in sorted({0, b - 1}):
            y = np.empty(V, dtype=dt)
            h.check(h.lib().hipMemcpy(y.ctypes.data, ctypes.c_void_p(arena.addr + int(o) + i * V * y.itemsize),
                                      y.nbytes, h.D2H), "hipMemcpy D2H")
            x = pools.host(s_, p)[first + i].reshape((1,) + s_).astype(np.complex128)
            key = "c128" if p == f.C128 else "c64"
            worst[key] = max(worst[key], _rel_l2(y.reshape((1,) + s_), _np_dft(x, d)))
    arena.close()
    return worst


def serving(pkg, n=20000, p99_cap_ms=2.0, streams=16, window_us=30.0):
    """Load test of the request server: the highest Poisson arrival rate whose p99 latency
    stays within p99_cap_ms, for continuous batching and for the two plain paths (one launch
    per request, each waited for; and the same with `streams` launches in flight), with a
    sampled check of each mode's results."""
    f, sv = pkg.fft3d, pkg.serving
    mix = sv.draw_mix(n, seed=0)
    pools = sv.InputPools(seed=0, keep_host=True)
    reqs = sv.make_requests(mix, pools, seed=1)
    req_bytes = sum(2 * r.batch * r.n0 * r.n1 * r.n2 * (16 if r.precision == 0 else 8)
                    for r in reqs) / n
    out = {"requests": n, "mean_io_bytes_per_request": req_bytes, "p99_cap_ms": p99_cap_ms,
           "budget_bytes": 64 << 30, "streams": streams, "window_us": window_us}
    modes = (("plain", f.SRV_PLAIN_SYNC), ("plain_async", f.SRV_PLAIN_ASYNC),
             ("batched", f.SRV_BATCHED))
    for mode, code in modes:
        srv = f.Server(budget_bytes=64 << 30, streams=streams, batched=code,
                       window_us=window_us if code == f.SRV_BATCHED else 0.0)
        ok, bad, pts = None, None, []
        rate = 4000.0
        while rate < 2e6:
            pt = sv.load_point(srv, reqs, rate)
            pts.append(pt)
            if pt["p99_ms"] <= p99_cap_ms:
                ok = pt
                rate *= 1.5
            else:
                bad = pt
                break
        if ok and bad:
            lo, hi = ok["rate"], bad["rate"]
            for _ in range(4):
                mid = 0.5 * (lo + hi)
                pt = sv.load_point(srv, reqs, mid)
                pts.append(pt)
                if pt["p99_ms"] <= p99_cap_ms:
                    ok, lo = pt, mid
                else:
                    hi = mid
        st = srv.stats()
        check = _serving_check(pkg, srv, pools)
        srv.close()
        out[mode] = dict(max_rate_req_s=ok["rate"] if ok else 0.0,
                         at_max=ok, stats=st, result_check_rel_l2=check,
                         points=[{k: round(v, 4) for k, v in p.items()} for p in pts])
        print(f"# serving {mode}: max rate {out[mode]['max_rate_req_s']:.0f}/s, check {check}",
              file=sys.stderr, flush=True)
    pools.close()
    ba = out["batched"]["at_max"]
    for mode in ("plain", "plain_async"):
        pl = out[mode]["at_max"]
        if pl and ba:
            out[f"throughput_ratio_vs_{mode}_at_p99_cap"] = (ba["transforms_per_s"] /
                                                            pl["transforms_per_s"])
    return out


LATENCY_CASES = [((6, 6, 6), -1), ((8, 8, 8), -1), ((12, 12, 12), -1), ((17, 17, 17), -1),
                 ((24, 24, 24), -1), ((36, 36, 36), -1)]


def small_batch_latency(pkg, reps=300):
    """Batch-1 complex128 executes: the device time per execute back to back (median of
    3 windows of >= 10 ms) and the host round trip of one execute followed by a stream
    synchronisation (median of `reps`), launched directly and replayed from a graph captured
    once per (in, out) pair (the reference replays graph execs for small batches,
    bench/gpu/impl_4/L17_dmma.cu:1002-1010)."""
    f, h = pkg.fft3d, pkg.hip
    out = {}
    for shape, d in LATENCY_CASES:
        V = shape[0] * shape[1] * shape[2]
        x = make_input(shape, 1, seed=5, dist="uniform")
        bi, bo = h.DeviceBuffer(16 * V), h.DeviceBuffer(16 * V)
        bi.upload(x)
        p = f.Plan(shape, 1, d, f.C128)
        s = h.Stream()
        g = h.GraphExec(s, lambda st: p.execute(bi.addr, bo.addr, stream=st))
        res = {"kernel": p.kernel}
        for mode, launch in (("direct", lambda: p.execute(bi.addr, bo.addr, stream=s)),
                             ("graph", lambda: g.launch(s))):
            for _ in range(20):
                launch()
            s.synchronize()
            rt = []
            for _ in range(reps):
                t0 = time.perf_counter()
                launch()
                s.synchronize()
                rt.append(time.perf_counter() - t0)
            e0, e1 = h.Event(), h.Event()
            e0.record(s)
            for _ in range(50):
                launch()
            e1.record(s)
            e1.synchronize()
            n = max(50, math.ceil(10.0 / (e0.elapsed_ms(e1) / 50)))
            evs = [h.Event() for _ in range(4)]
            evs[0].record(s)
            for w in range(3):
                for _ in range(n):
                    launch()
                evs[w + 1].record(s)
            evs[-1].synchronize()
            ws = sorted(evs[w].elapsed_ms(evs[w + 1]) / n * 1e3 for w in range(3))
            for e in evs + [e0, e1]:
                e.close()
            res[mode] = dict(device_us_per_execute=ws[1],
                             round_trip_us_median=float(np.median(rt)) * 1e6,
                             round_trip_us_p99=float(np.percentile(rt, 99)) * 1e6)
        y = bo.download(np.complex128, x.shape)
        res["rel_l2_vs_numpy"] = _rel_l2(y, _np_dft(x, d))
        g.close()
        p.close()
        s.close()
        bi.close()
        bo.close()
        out["x".join(map(str, shape))] = res
    return out


def host_abi(pkg, L=17, batch=1024, reps=8):
    """The reference's host-pointer ABI (fft3d_create / fft3d_execute, bench/geom/fft3d_api.h)
    on this library at the headline size: each execute copies the batch in from pageable host
    memory, transforms it and copies it back before returning, as bench/geom/driver.c
    requires, so its rate is bounded by the host side and the host link, not HBM.  Median
    of `reps` executes after one warm-up, output checked against numpy.fft."""
    f = pkg.fft3d
    L_ = f.load()
    x = make_input((L, L, L), batch, seed=9, dist="uniform")
    y = np.empty_like(x)
    h = L_.fft3d_create(L, batch)
    if not h:
        return None
    try:
        L_.fft3d_execute(h, x.ctypes.data, y.ctypes.data)
        ts = []
        for _ in range(reps):
            t0 = time.perf_counter()
            L_.fft3d_execute(h, x.ctypes.data, y.ctypes.data)
            ts.append(time.perf_counter() - t0)
    finally:
        L_.fft3d_destroy(h)
    t = float(np.median(ts))
    return {"L": L, "batch": batch, "ms_per_execute": t * 1e3, "transforms_per_s": batch / t,
            "host_link_GBs_each_way": x.nbytes / t / 1e9,
            "rel_l2_vs_numpy": _rel_l2(y, _np_dft(x, -1)),
            "note": "pageable host buffers: copies into pinned staging, H2D, transform, D2H "
                    "and copies out per execute, pipelined in ~8 MB chunks; not `value`"}


# What the printed line keeps of each block.
BRIEF = {
    "cpu_baseline": ("value", "unit", "cores", "kind", "sample"),
    "secondary": ("kernel", "ms_per_execute", "transforms_per_s", "roofline_frac", "rel_l2_vs_numpy"),
    "precision_variants": ("kernel", "us", "rel_l2"),
    "small_batch_latency": ("kernel", "device_us_per_execute", "round_trip_us_median"),
    "host_abi": ("ms_per_execute", "transforms_per_s", "rel_l2_vs_numpy"),
    "serving": ("max_rate_req_s", "p50_ms", "p99_ms", "transforms_per_s", "c128", "c64",
                "throughput_ratio_vs_plain_at_p99_cap", "throughput_ratio_vs_plain_async_at_p99_cap"),
}


def brief(record):
    """The printed line: the record with the blocks of BRIEF cut to the leaves named there (at any
    depth) and their figures to five digits."""
    def cut(v, keys):
        if isinstance(v, dict):
            kept = {k: cut(x, keys) for k, x in v.items()
                    if k in keys or isinstance(x, dict)}
            return {k: x for k, x in kept.items() if x != {}}
        return float(f"{v:.5g}") if isinstance(v, float) else v
    return {k: cut(v, BRIEF[k]) if k in BRIEF and v is not None else v for k, v in record.items()}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--windows", type=int, default=5,
                    help="timed windows after the contract region (the value is their median)")
    ap.add_argument("--window-ms", type=float, default=20.0, help="minimum window length")
    ap.add_argument("--record", default=None, metavar="PATH", help="write the full record there")
    ap.add_argument("--no-secondary", action="store_true")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-serving", action="store_true")
    ap.add_argument("--no-precision", action="store_true")
    ap.add_argument("--no-latency", action="store_true")
    ap.add_argument("--workload", default=None,
                    help="time only this secondary workload (e.g. L8_c128_fwd_b4096) and print "
                         "its measurement; for profiling runs, no JSON line")
    a = ap.parse_args()
    if a.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) > 1:
        print("bench.py: measures one GPU only; batches of independent volumes "
              "shard across GPUs with no communication.", file=sys.stderr)
        sys.exit(2)
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    # The CPU baseline spawns the reference binaries, so it runs before HIP is initialised.
    cpu = None if a.no_cpu else cpu_baseline()
    if cpu:
        print(f"# cpu_baseline: {cpu}", file=sys.stderr, flush=True)
    import __graft_entry__
    pkg = __graft_entry__.load_package()
    if pkg.hip.device_count() < 1:
        print("bench.py: no HIP device", file=sys.stderr)
        sys.exit(1)
    pkg.hip.check(pkg.hip.lib().hipSetDevice(0), "hipSetDevice")

    if a.workload:
        wl = [w for w in SECONDARY if w["name"] == a.workload]
        if not wl:
            print(f"bench.py: unknown workload {a.workload}", file=sys.stderr)
            sys.exit(2)
        print(f"# {a.workload}: {measure(pkg, wl[0], a.steps, a.warmup, windows=a.windows, window_ms=a.window_ms)}", flush=True)
        return
    head = measure(pkg, HEADLINE, a.steps, a.warmup, windows=a.windows, window_ms=a.window_ms)
    print(f"# headline {HEADLINE['name']}: {head}", file=sys.stderr, flush=True)
    secondary = {}
    if not a.no_secondary:
        for wl in SECONDARY:
            secondary[wl["name"]] = measure(pkg, wl, max(10, a.steps // 2), a.warmup,
                                            windows=a.windows, window_ms=a.window_ms)
            print(f"# {wl['name']}: {secondary[wl['name']]}", file=sys.stderr, flush=True)
    precision = None if a.no_precision else precision_mix(pkg)
    if precision:
        print(f"# precision variants: {precision}", file=sys.stderr, flush=True)
    latency = None if a.no_latency else small_batch_latency(pkg)
    if latency:
        print(f"# batch-1 latency: {latency}", file=sys.stderr, flush=True)
    serve = None if a.no_serving else serving(pkg)
    habi = None if a.no_latency else host_abi(pkg)
    if habi:
        print(f"# host ABI: {habi}", file=sys.stderr, flush=True)
    V = 17 ** 3
    line = {
        "metric": "batched transforms/s + % HBM roofline at L=8/17/36 fp64; serving p99 latency",
        "value": head["transforms_per_s"],
        "unit": "transforms/s",
        "n_gpus": 1,
        "steps": a.steps,
        "warmup": a.warmup,
        "ms_per_step": head["ms_per_execute"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64",
        "data": "synthetic: iid uniform(-1,1) real and imaginary parts, seeded",
        "config": {"workload": "17x17x17 complex128 forward 3D FFT, batch 1024, "
                               "device-resident, rotated buffers",
                   "n0": 17, "n1": 17, "n2": 17, "batch": 1024, "precision": "complex128",
                   "direction": "forward", "kernel": head["kernel"],
                   "rotate_pairs": head["rotate_pairs"]},
        "gflops_nominal": 5.0 * V * math.log2(V) * head["transforms_per_s"] / 1e9,
        "rel_l2_vs_numpy": head["rel_l2_vs_numpy"],
        "roofline": {"bound": "hbm", "achieved": head["achieved_GBs"], "peak": PEAK_HBM_GBS,
                     "unit": "GB/s", "frac": head["roofline_frac"],
                     "traffic": TRAFFIC if head["kernel"] == TRAFFIC_KERNEL else None,
                     "traffic_source": "rocprofv3 FETCH_SIZE + WRITE_SIZE of this kernel at "
                                       "this workload, copy-calibrated, from the committed "
                                       "profile (not measured in this run)",
                     "kernel_us_mean": head["ms_per_execute"] * 1e3,
                     "algorithmic_bytes_per_launch": head["algorithmic_bytes_per_execute"]},
        "timing": {k: head[k] for k in ("windows", "executes_per_window", "window_ms",
                                        "window_spread", "us_per_execute_min",
                                        "us_per_execute_max", "contract_ms_total",
                                        "contract_ms_per_execute")},
        "cpu_baseline": cpu,
        "secondary": secondary,
        "precision_variants": precision,
        "small_batch_latency": latency,
        "host_abi": habi,
        "serving": serve,
    }
    if a.record:
        with open(a.record, "w") as out:
            json.dump(line, out, indent=1)
    print(json.dumps(brief(line)), flush=True)


if __name__ == "__main__":
    main()
