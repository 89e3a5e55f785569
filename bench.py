#!/usr/bin/env python3
"""Benchmark of the hot path on one MI355X: the kernels of cuTile.jl's examples, through the
C ABI of libmi355tile.so.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--kernels LIST|all|none] [--no-cpu] [--table]
    (--kernels gemm_shapes: opt-in sweep of the GEMM entry points over other shapes, not part of 'all')

The LAST line of stdout is one small JSON record (under 4 KB: the contract keys, ``roofline``, ``cpu_baseline`` and a
compact ``summary`` of every north-star figure); the full record with one entry per kernel, the achieved errors and
the per-stage times goes to ``--detail-file`` (default gpurun_out/bench_full.json) and, with ``--full``, to an
earlier stdout line.  A "step" is one pass of the headline workload over one batch
of synthetic, seeded input already resident in HBM:

    headline workload = the second of the benchmark configurations: row LayerNorm fwd + bwd
    (y, dx, dgamma, dbeta) and the row softmax on 4096x4096 fp32.
    ``value`` = algorithmic bytes of the step / wall time per step, in GB/s, timed over
    exactly ``--steps`` steps between two device synchronisations.

Every other configuration (vadd, transpose, GEMM, batched GEMM, FMHA, MoE f16 and fp8, and the
follow-up rows: FFT, Tiled broadcast / mapreduce, RNG fills) is measured in the same run and reported
under ``"kernels"`` of the full record:
  * ``min_ms`` / ``mean_ms``: the reference's protocol (examples/benchmarks.jl:12-13: 5 warm-up
    launches, 20 launches each bracketed by its own pair of events on the launch stream);
  * ``avg_ms``: 20 launches back to back between ONE pair of events (no per-launch event
    and host overhead; this is what agrees with a profiler's average kernel duration);
  * ``achieved`` (from ``avg_ms``) in GB/s or TFLOP/s and ``frac`` of the MI355X roofline
    (HBM 8 TB/s; dense MFMA f16 2.5 PFLOP/s, fp8 5.0 PFLOP/s, fp32 157.3 TFLOP/s);
  * ``cpu_ms``: the numpy/OpenBLAS restatement of the reference's CPU path for the same
    configuration (or a stated sample of it), timed on this host.
The top-level ``roofline`` is the dominant kernel of the headline workload, with its average
launch duration measured by one pair of events per step inside the timed region (``stages_ms``
comes from a second, untimed pass with events between all stages); ``cpu_baseline`` is the CPU
restatement of the headline workload on a bounded sample.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
NRUNS, WARMUP = 20, 5  # examples/benchmarks.jl:12-13


def _event_times(fn, nruns, warmup):
    """Reference protocol: each launch bracketed by its own events; returns ms per launch."""
    import torch
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    out = []
    for _ in range(nruns):
        e0 = torch.cuda.Event(enable_timing=True); e1 = torch.cuda.Event(enable_timing=True)
        e0.record(); fn(); e1.record(); e1.synchronize()
        out.append(e0.elapsed_time(e1))
    return out


WARM_MS, TIMED_MS = 5.0, 20.0   # GPU time of the untimed launches in front of a timed batch, and of the batch itself


def _batch_counts(nruns, est_ms):
    if not est_ms:
        return nruns, nruns
    return max(nruns, min(1000, int(WARM_MS / est_ms))), max(nruns, min(4000, int(TIMED_MS / est_ms)))


def _back_to_back(fn, nruns, est_ms=None):
    """A batch of launches between one pair of events; returns average ms per launch.  With an estimate of the
    launch duration the batch lasts about TIMED_MS of GPU time (never fewer than nruns launches) and stands
    directly behind about WARM_MS of untimed launches of the same kernel, so that it runs at the clocks of a
    busy GPU: coming from idle, the power management takes milliseconds to settle (the attention kernel takes
    31-33 us per launch in bursts of 20 to 200 launches from idle and 28.5 us in a run of 2000; the f16 GEMM,
    which is power-limited, moves the other way)."""
    import torch
    torch.cuda.synchronize()
    e0 = torch.cuda.Event(enable_timing=True); e1 = torch.cuda.Event(enable_timing=True)
    warm, n = _batch_counts(nruns, est_ms)
    for _ in range(warm):
        fn()
    e0.record()
    for _ in range(n):
        fn()
    e1.record(); e1.synchronize()
    return e0.elapsed_time(e1) / n


def _entry(name, fn, work, unit, bound, peak, dtype, nruns, warmup, extra=None, cold=None):
    """``cold``: a list of launches of the same kernel on distinct buffer sets, enough of them that more than
    the 256 MB memory-side cache holds is touched between two uses of a set; ``frac_cold`` is measured
    by cycling through them, so that no launch finds its input resident."""
    calls = [0]
    raw_fn = fn

    def fn():
        calls[0] += 1
        return raw_fn()
    t = _event_times(fn, nruns, warmup)
    batches = [_back_to_back(fn, nruns, min(t)) for _ in range(2)]
    avg = min(batches)   # best of two batches: a one-off stall does not define the rate
    scale = 1e9 if unit == "GB/s" else 1e12
    ach = work / (avg * 1e-3) / scale
    e = {"name": name, "min_ms": round(min(t), 5), "mean_ms": round(sum(t) / len(t), 5), "avg_ms": round(avg, 5),
         "avg_ms_is": "best of 2 batches of %d back-to-back launches (about %.0f ms), each directly behind %d untimed ones" % (_batch_counts(nruns, min(t))[1], TIMED_MS, _batch_counts(nruns, min(t))[0]),
         "work": work, "achieved": round(ach, 2), "unit": "GB/s" if unit == "GB/s" else "TFLOP/s", "bound": bound,
         "peak": peak, "frac": round(ach / peak, 4), "dtype": dtype}
    e["launches"] = calls[0]   # calls of the entry point made for the figures above (warm-up included)
    if cold:
        k = len(cold)

        def cycle():
            for f in cold:
                f()
        cycle()
        # (batches as long as the warm ones and behind as many untimed launches: three cycles from an idle GPU ran at
        # the clocks of the ramp, 8-15 % below what the same rotation reaches once they have settled)
        cavg = min(_back_to_back(cycle, max(1, nruns // k), k * min(t)) for _ in range(2)) / k
        e["avg_ms_cold"] = round(cavg, 5)
        e["frac_cold"] = round(work / (cavg * 1e-3) / scale / peak, 4)
        e["cold_sets"] = k
    if extra:
        e.update(extra)
    return e


def _shader_clock_mhz():
    """Current shader clock from the driver's sysfs table (the level marked '*'), or None."""
    import glob
    best = None
    for path in glob.glob("/sys/class/drm/card*/device/pp_dpm_sclk"):
        try:
            for line in open(path):
                if "*" in line:
                    mhz = int("".join(ch for ch in line.split(":")[1] if ch.isdigit()))
                    best = mhz if best is None else max(best, mhz)
        except Exception:
            pass
    return best


def _clock_under_load(fn, seconds=0.25):
    """Keep ``fn`` queued for about ``seconds`` and sample the shader clock meanwhile; MHz (median) or None."""
    import torch
    samples = []
    t0 = time.perf_counter()
    while time.perf_counter() - t0 < seconds:
        for _ in range(8):
            fn()
        c = _shader_clock_mhz()
        if c is not None:
            samples.append(c)
        torch.cuda.synchronize()
    samples.sort()
    return samples[len(samples) // 2] if samples else None


def _cpu_time(fn, repeats=3):
    fn()  # warm-up
    best = float("inf")
    for _ in range(repeats):
        t0 = time.perf_counter(); fn(); best = min(best, time.perf_counter() - t0)
    return best * 1e3


def bench_kernels(ct, which, cpu, nruns=NRUNS, warmup=WARMUP):
    """Measure each configuration; returns {key: entry}."""
    import numpy as np
    import torch
    from oracle import cutile_oracle as orc
    from cutile_jl_amd.examples import vadd, transpose, layernorm, softmax, matmul, batchmatmul, fmha, moe, fft
    res = {}
    ncores = os.cpu_count()

    def want(n):
        return which is None or n in which

    if want("vadd"):
        d = vadd.prepare(benchmark=True)
        A, B, C = ct.TileArray(d.a), ct.TileArray(d.b), ct.TileArray(d.c)
        e = _entry("vadd 2^27 f32", lambda: ct.vec_add_kernel_1d(A, B, C, 1024), vadd.metric(d)[0], "GB/s", "hbm",
                   HBM_PEAK_GBS, "f32", nruns, warmup, {"variant": None})
        e["variant"] = ct.last_variant()
        if cpu:
            a, b = d.a.cpu().numpy(), d.b.cpu().numpy()
            e["cpu_ms"] = round(_cpu_time(lambda: a + b), 2); e["cpu_note"] = "numpy a+b, 1 thread"
        res["vadd"] = e
        del d
    if want("transpose"):
        d = transpose.prepare(benchmark=True)
        X, Y = ct.TileArray(d.x), ct.TileArray(d.y)
        e = _entry("transpose 8192^2 f32", lambda: ct.transpose_kernel(X, Y, 64, 64), transpose.metric(d)[0], "GB/s",
                   "hbm", HBM_PEAK_GBS, "f32", nruns, warmup)
        e["variant"] = ct.last_variant()
        if cpu:
            x = d.x.cpu().numpy()
            e["cpu_ms"] = round(_cpu_time(lambda: np.ascontiguousarray(x.T)), 2); e["cpu_note"] = "numpy transpose copy, 1 thread"
        res["transpose"] = e
        del d
    if want("layernorm"):
        for G in (64, 256):
            sets = [layernorm.prepare(benchmark=True, GROUP_SIZE_M=G, seed=1 + i) for i in range(6 if G == 64 else 1)]
            d = sets[0]
            MN4 = d.M * d.N * 4

            def launches(dd):
                D = {k: ct.TileArray(getattr(dd, k)) for k in ("X", "W", "B", "Y", "Mean", "Rstd", "DY", "DX", "DW_partial",
                                                                "DB_partial", "Locks", "FINAL_DW", "FINAL_DB")}

                def fwd():
                    ct.layer_norm_fwd(D["X"], D["W"], D["B"], D["Y"], D["Mean"], D["Rstd"], dd.eps, 1024)

                def bwd():
                    dd.partials.zero_()
                    ct.layer_norm_bwd_dx_partial_dwdb(D["DX"], D["DY"], D["DW_partial"], D["DB_partial"], D["X"], D["W"],
                                                      D["Mean"], D["Rstd"], D["Locks"], G, 1024)
                    ct.layer_norm_bwd_dwdb(D["DW_partial"], D["DB_partial"], D["FINAL_DW"], D["FINAL_DB"], 32, 1024)
                def bwd_static():   # the same backward with the slots in the library's own array: two launches, no fill
                    ct.layer_norm_bwd_static(dd.DX, dd.DY, dd.X, dd.W, dd.Mean, dd.Rstd, dd.FINAL_DW, dd.FINAL_DB, G, 32, 1024)
                fwd._keep = D
                return fwd, bwd, bwd_static

            fb = [launches(dd) for dd in sets]
            fwd, bwd, bwd_static = fb[0]
            for f, _, _ in fb:
                f()     # Mean / Rstd of every set, for its backward
            fwd_bytes = 2 * MN4 + (2 * d.N + 2 * d.M) * 4
            bwd_bytes = 3 * MN4 + (d.N + 2 * d.M) * 4 + 4 * d.N * G * 4 + 2 * d.N * 4
            if G == 64:
                res["layernorm_fwd"] = _entry("LayerNorm fwd 4096^2 f32", fwd, fwd_bytes, "GB/s", "hbm", HBM_PEAK_GBS,
                                              "f32", nruns, warmup, {"reference_formula_bytes": 4 * MN4},
                                              cold=[f for f, _, _ in fb])
                fwd(); res["layernorm_fwd"]["variant"] = ct.last_variant()
            key = "layernorm_bwd" if G == 64 else "layernorm_bwd_G256"
            res[key] = _entry(f"LayerNorm bwd 4096^2 f32, GROUP_SIZE_M={G} (1 fill + 2 kernels)", bwd, bwd_bytes,
                              "GB/s", "hbm", HBM_PEAK_GBS, "f32", nruns, warmup, {"reference_formula_bytes": 5 * MN4},
                              cold=[b for _, b, _ in fb] if G == 64 else None)
            if G == 64:
                res["layernorm_bwd_static"] = _entry("LayerNorm bwd 4096^2 f32, GROUP_SIZE_M=64, slots in the library's array (2 kernels, no fill)",
                                                     bwd_static, bwd_bytes, "GB/s", "hbm", HBM_PEAK_GBS, "f32", nruns, warmup,
                                                     cold=[b for _, _, b in fb])
            if cpu and G == 64:
                X, W, B, DY = (orc.to_julia(t) for t in (d.X, d.W, d.B, d.DY))
                sub = slice(0, 512)
                res["layernorm_fwd"]["cpu_ms"] = round(_cpu_time(lambda: orc.layer_norm_fwd(X[:, sub], W, B, d.eps, dtype=np.float32)) * 8, 1)
                res["layernorm_fwd"]["cpu_note"] = "numpy 1 thread, 512 of 4096 rows x8"
                res[key]["cpu_ms"] = round(_cpu_time(lambda: orc.layer_norm_bwd(X[:, sub], W, DY[:, sub], d.eps, dtype=np.float32)) * 8, 1)
                res[key]["cpu_note"] = "numpy 1 thread, 512 of 4096 rows x8"
            del d, sets, fb, fwd, bwd, bwd_static
    if want("softmax"):
        sets = [softmax.prepare(benchmark=True, seed=2 + i) for i in range(6)]
        d = sets[0]
        MN4 = d.M * d.N * 4
        tma, chk = [], []
        for dd in sets:
            I, O1, O2 = ct.TileArray(dd.input), ct.TileArray(dd.output_tma), ct.TileArray(dd.output_chunked)
            tma.append((lambda I=I, O1=O1: ct.softmax_tma_kernel(O1, I, 4096, d.M)))
            chk.append((lambda I=I, O2=O2: ct.softmax_chunked_kernel(O2, I, d.N, 1024, d.M)))
        res["softmax_tma"] = _entry("softmax (single tile) 4096^2 f32", tma[0],
                                    2 * MN4, "GB/s", "hbm", HBM_PEAK_GBS, "f32", nruns, warmup, cold=tma)
        res["softmax_tma"]["variant"] = ct.last_variant()
        res["softmax_chunked"] = _entry("softmax (chunked) 4096^2 f32", chk[0], 2 * MN4, "GB/s", "hbm",
                                        HBM_PEAK_GBS, "f32", nruns, warmup, {"reference_formula_bytes": 4 * MN4}, cold=chk)
        if cpu:
            x = orc.to_julia(d.input)
            res["softmax_tma"]["cpu_ms"] = round(_cpu_time(lambda: orc.softmax(x[:, :512], dtype=np.float32)) * 8, 1)
            res["softmax_tma"]["cpu_note"] = "numpy 1 thread, 512 of 4096 columns x8"
        del d, sets, tma, chk
    if want("copy_ref"):
        # Yardstick for the 64 MB row kernels: a plain 64 MB -> 64 MB copy (the generated Tiled(Y) .= Tiled(X)
        # kernel) on resident buffers and cycling over six buffer pairs.  What it reaches cold is the ceiling of
        # any one-pass row kernel of this size on cold input.
        from cutile_jl_amd import tiled as T
        n = 1 << 24
        pairs = [(torch.rand(n, device="cuda"), torch.empty(n, device="cuda")) for _ in range(6)]
        fns = [(lambda x=x, y=y: T.Tiled(y).assign(T.Tiled(x))) for x, y in pairs]
        res["copy_ref"] = _entry("yardstick: copy 64 MB -> 64 MB f32 (Tiled(Y) .= Tiled(X))", fns[0], 8 * n, "GB/s", "hbm",
                                 HBM_PEAK_GBS, "f32", nruns, warmup, cold=fns)
        # The same yardstick from code that is not this library's: the runtime's device-to-device copy
        # (torch's copy_ of a contiguous tensor is hipMemcpyAsync) over the same six buffer pairs.
        rfns = [(lambda x=x, y=y: y.copy_(x)) for x, y in pairs]
        res["copy_ref_runtime"] = _entry("yardstick: copy 64 MB -> 64 MB f32 (runtime device-to-device copy)", rfns[0], 8 * n, "GB/s",
                                         "hbm", HBM_PEAK_GBS, "f32", nruns, warmup, cold=rfns)
        del pairs, fns, rfns
    if want("matmul"):
        d = matmul.prepare(benchmark=True, T=torch.float16, out_T=torch.float32, dist="normal64")
        A, B, C = ct.TileArray(d.A), ct.TileArray(d.B), ct.TileArray(d.C)
        e = _entry("GEMM 4096^3 f16 -> f32", lambda: ct.matmul_kernel(A, B, C, 64, 64, 64), matmul.metric(d)[0],
                   "TFLOPS", "mfma", 2500.0, "f16", nruns, warmup)
        e["variant"] = ct.last_variant()
        e["shader_clock_mhz"] = _clock_under_load(lambda: ct.matmul_kernel(A, B, C, 64, 64, 64))
        if cpu:
            a = orc.to_julia(d.A).astype(np.float32); b = orc.to_julia(d.B).astype(np.float32)
            e["cpu_ms"] = round(_cpu_time(lambda: a @ b, repeats=2), 1); e["cpu_note"] = f"numpy/OpenBLAS sgemm on widened inputs, {ncores} threads"
        res["matmul"] = e
        del d
    if want("matmul_fp8"):
        # fp8 x fp8 operands (ext/DLFP8TypesExt.jl:15-19): the same 4096^3 problem on the fp8 matrix cores
        g = torch.Generator().manual_seed(6)
        for key, T8, nm in (("matmul_fp8", torch.float8_e4m3fn, "e4m3fn"), ("matmul_fp8_e5m2", torch.float8_e5m2, "e5m2")):
            a8 = torch.randn(4096, 4096, generator=g).to(T8).cuda(); b8 = torch.randn(4096, 4096, generator=g).to(T8).cuda()
            c8 = torch.empty(4096, 4096, device="cuda")
            A, B, C = ct.TileArray(a8), ct.TileArray(b8), ct.TileArray(c8)
            e = _entry(f"GEMM 4096^3 {nm} x {nm} -> f32 (inputs ~ N(0,1) rounded to fp8)", lambda: ct.matmul_kernel(A, B, C, 64, 64, 64),
                       2.0 * 4096 ** 3, "TFLOPS", "mfma", 5000.0, "fp8", nruns, warmup)
            e["variant"] = ct.last_variant()
            e["shader_clock_mhz"] = _clock_under_load(lambda: ct.matmul_kernel(A, B, C, 64, 64, 64))
            res[key] = e
            del a8, b8, c8
    if which is not None and "gemm_shapes" in which:
        # Opt-in (not part of 'all'): the same entry points at other shapes, among them the size lists of the
        # reference examples' main() (matmul.jl:156-165, batchmatmul.jl:161-169), shapes off the tile grid and
        # problems with few tiles, where the direct-to-LDS kernels switch to 256x128 / 128x128 tiles.
        shapes = [("f16", 1, 256, 256, 256), ("f16", 1, 512, 512, 512), ("f16", 1, 1024, 1024, 1024), ("f16", 1, 2048, 2048, 2048),
                  ("f16", 1, 2560, 2560, 2560), ("f16", 1, 3072, 3072, 3072), ("f16", 1, 4096, 2048, 4096), ("f16", 1, 4000, 4000, 4000),
                  ("f16", 1, 4096, 4096, 4000), ("f16", 1, 8192, 8192, 8192), ("f16", 4, 512, 1024, 256),
                  ("f32", 1, 256, 256, 256), ("f32", 1, 512, 512, 512), ("f32", 1, 256, 512, 128), ("f32", 1, 1024, 1024, 1024),
                  ("f32", 1, 2048, 2048, 2048), ("f32", 1, 4096, 4096, 4096), ("f32", 4, 256, 256, 128), ("f32", 4, 512, 512, 256),
                  # dense operands whose rows are not 16-byte aligned / sizes that are not multiples of a 16-byte vector
                  ("f16", 1, 4095, 4096, 4096), ("f16", 1, 4096, 4096, 4095), ("f16", 1, 4095, 4095, 4095), ("f16", 1, 4097, 4096, 4100),
                  ("f16", 1, 2047, 2048, 200), ("f32", 1, 4095, 4095, 4095),
                  ("e4m3", 1, 4096, 4096, 4096), ("e4m3", 1, 4095, 4096, 4096), ("e4m3", 1, 4096, 4096, 4095), ("e4m3", 1, 4095, 4095, 4095)]
        rows = []
        for (dt, Bt, M, N, K) in shapes:
            T = {"f16": torch.float16, "f32": torch.float32, "e4m3": torch.float8_e4m3fn}[dt]
            a = (torch.randn(Bt, K, M, device="cuda") / 8).to(T); b = (torch.randn(Bt, N, K, device="cuda") / 8).to(T)
            c = torch.empty(Bt, N, M, device="cuda", dtype=torch.float32)
            if Bt == 1:
                A, B, C = ct.TileArray(a[0]), ct.TileArray(b[0]), ct.TileArray(c[0])
                fn = lambda: ct.matmul_kernel(A, B, C, 64, 64, 64)
            else:
                A, B, C = ct.TileArray(a), ct.TileArray(b), ct.TileArray(c)
                fn = lambda: ct.batch_matmul_kernel(A, B, C, 64, 64, 64)
            e = _entry(f"GEMM {dt} batch {Bt} M={M} N={N} K={K}", fn, 2.0 * Bt * M * N * K, "TFLOPS", "mfma",
                       {"f16": 2500.0, "f32": 157.3, "e4m3": 5000.0}[dt], dt, nruns, warmup)
            e["variant"] = ct.last_variant()
            rows.append(e)
        res["gemm_shapes"] = {"name": "GEMM at other shapes (opt-in)", "rows": rows}
    if want("batchmatmul"):
        d = batchmatmul.prepare(benchmark=True)
        A, B, C = ct.TileArray(d.A), ct.TileArray(d.B), ct.TileArray(d.C)
        e = _entry("batched GEMM 8x(1024x512x2048) f32", lambda: ct.batch_matmul_kernel(A, B, C, 128, 128, 64),
                   batchmatmul.metric(d)[0], "TFLOPS", "mfma", 157.3, "f32", nruns, warmup)
        e["variant"] = ct.last_variant()
        e["shader_clock_mhz"] = _clock_under_load(lambda: ct.batch_matmul_kernel(A, B, C, 128, 128, 64))
        if cpu:
            a = orc.to_julia(d.A); b = orc.to_julia(d.B)
            e["cpu_ms"] = round(_cpu_time(lambda: orc.batch_matmul(a, b, dtype=np.float32), repeats=2), 1)
            e["cpu_note"] = f"numpy/OpenBLAS sgemm per batch, {ncores} threads"
        res["batchmatmul"] = e
        del d
    if want("fmha"):
        d = fmha.prepare(benchmark=True)
        out = torch.empty_like(d.Q)
        Q, K, V, O = (ct.TileArray(t) for t in (d.Q, d.K, d.V, out))
        scale = float(np.float32(1.0 / np.sqrt(d.d_k)))
        e = _entry("causal FMHA 8x16x1024x64 f16",
                   lambda: ct.fmha_kernel(Q, K, V, O, scale, 0, d.d_k, d.heads, 128, 128, 1, True, True),
                   fmha.causal_flops(d), "TFLOPS", "mfma", 2500.0, "f16", nruns, warmup)
        e["variant"] = ct.last_variant()
        e["dense_count_flop"] = fmha.metric(d)[0]
        e["tflops_dense_count"] = round(fmha.metric(d)[0] / (e["avg_ms"] * 1e-3) / 1e12, 2)
        # the reference's timed region is cutile_fmha, which allocates Out (fmha.jl:160,265-267)
        with_alloc = lambda: fmha.cutile_fmha(d.Q, d.K, d.V, causal=True)
        with_alloc()
        e["avg_ms_with_out_alloc"] = round(min(_back_to_back(with_alloc, nruns) for _ in range(2)), 5)
        e["shader_clock_mhz"] = _clock_under_load(lambda: ct.fmha_kernel(Q, K, V, O, scale, 0, d.d_k, d.heads, 128, 128, 1, True, True))
        if cpu:
            q, k, v = (orc.to_julia(t)[:, :, :, :1] for t in (d.Q, d.K, d.V))
            e["cpu_ms"] = round(_cpu_time(lambda: orc.ref_fmha(q[:, :, :4], k[:, :, :4], v[:, :, :4], causal=True), repeats=2) * 32, 1)
            e["cpu_note"] = f"numpy restatement of ref_fmha, 4 of 128 (batch, head) pairs x32, BLAS {ncores} threads"
        res["fmha"] = e
        del d
        # The same entry point on the other end of its argument range (input_pos, fmha.jl:45-46): one new token per
        # sequence against a cache of 4096 keys.  Bound by reading the cache once.
        # (the third: a cache of 537 MB, twice what the memory-side cache holds, i.e. keys that really come from HBM at
        # every launch; the library requests those with non-temporal transfers)
        for key, (B, H, G, Skv) in (("fmha_decode", (8, 16, 1, 4096)), ("fmha_decode_grouped", (32, 32, 4, 2048)),
                                    ("fmha_decode_16k", (8, 16, 1, 16384))):
            dd = fmha.prepare(batch=B, heads=H, seq_q=1, seq_kv=Skv, query_group_size=G, causal=True)
            od = torch.empty_like(dd.Q)
            Qd, Kd, Vd, Od = (ct.TileArray(t) for t in (dd.Q, dd.K, dd.V, od))
            go = lambda: ct.fmha_kernel(Qd, Kd, Vd, Od, scale, Skv - 1, 64, H, 128, 128, G, True, True)
            go()
            nb = (dd.K.numel() + dd.V.numel() + 2 * dd.Q.numel()) * 2
            ed = _entry(f"FMHA decode: 1 query per sequence at input_pos = {Skv - 1}, {B}x{H} heads in groups of {G}, {Skv} cached keys, f16 "
                        "(keys split over workgroups, the last part to arrive adds the parts: one launch)", go, nb, "GB/s", "hbm", HBM_PEAK_GBS, "f16", nruns, warmup)
            ed["variant"] = ct.last_variant()
            res[key] = ed
            del dd
    if want("fft"):
        d = fft.prepare(benchmark=True)
        F0, F1, F2 = d.factors
        go = ct.bind("mi_fft_kernel", d.x_packed, d.y_packed, d.W0, d.W1, d.W2, d.T0, d.T1, d.N, F0, F1, F2, 1, d.D)
        nbytes = 2 * d.batch * d.N * 8 + (d.T0.numel() + d.T1.numel() + d.W0.numel() * 3) * 4
        res["fft"] = _entry("FFT 4096-point x 256 signals complex64 (3-stage 16x16x16), latency benchmark of the reference",
                            go, nbytes, "GB/s", "hbm", HBM_PEAK_GBS, "f32", nruns, warmup)
        if cpu:
            x = d.input.cpu().numpy()
            res["fft"]["cpu_ms"] = round(_cpu_time(lambda: np.fft.fft(x, axis=1)), 2)
            res["fft"]["cpu_note"] = "numpy.fft (pocketfft) on the same complex64 batch, 1 thread (the reference verifies against FFTW)"

    if want("tiled"):
        # Host-level Tiled broadcast / mapreduce (src/broadcast.jl, src/mapreduce.jl): kernels generated at run time.
        from cutile_jl_amd import tiled as T
        n = 1 << 27
        A = torch.rand(n, device="cuda"); B = torch.rand(n, device="cuda"); C = torch.empty(n, device="cuda")
        M, Cm = A.view(8192, 16384), C.view(8192, 16384)          # Julia (16384, 8192)
        row = torch.rand(8192, 1, device="cuda")                  # Julia (1, 8192)
        legs = [
            ("tiled_broadcast_add", "Tiled(C) .= Tiled(A) .+ Tiled(B), 2^27 f32", lambda: T.Tiled(C).assign(T.Tiled(A) + T.Tiled(B)), 12 * n),
            ("tiled_broadcast_fused", "Tiled(C) .= A .+ A .* sin.(B), 2^27 f32, one fused kernel",
             lambda: T.Tiled(C).assign(T.Tiled(A) + T.Tiled(A) * T.sin(T.Tiled(B))), 12 * n),
            ("tiled_broadcast_expand", "Tiled(C) .= M .+ row, M (16384, 8192), row (1, 8192) f32", lambda: T.Tiled(Cm).assign(T.Tiled(M) + T.Tiled(row)), 8 * n),
            ("tiled_sum_all", "sum(Tiled(A); dims=1), 2^27 f32 (two passes)", lambda: T.sum(T.Tiled(A), dims=1), 4 * n),
            ("tiled_sum_dims1", "sum(Tiled(M); dims=1), (16384, 8192) f32: contiguous runs", lambda: T.sum(T.Tiled(M), dims=1), 4 * n),
            ("tiled_sum_dims2", "sum(Tiled(M); dims=2), (16384, 8192) f32: strided (two passes)", lambda: T.sum(T.Tiled(M), dims=2), 4 * n),
            ("tiled_maximum_dims2", "maximum(Tiled(M); dims=2), NaN-propagating", lambda: T.maximum(T.Tiled(M), dims=2), 4 * n),
        ]
        for key, name, fn, nbytes in legs:
            res[key] = _entry(name, fn, nbytes, "GB/s", "hbm", HBM_PEAK_GBS, "f32", nruns, warmup)
            res[key]["variant"] = ct.last_variant()
        if cpu:
            a, b = A[: n // 16].cpu().numpy(), B[: n // 16].cpu().numpy()
            res["tiled_broadcast_fused"]["cpu_ms"] = round(_cpu_time(lambda: a + a * np.sin(b)) * 16, 1)
            res["tiled_broadcast_fused"]["cpu_note"] = "numpy a + a*sin(b) on 1/16 of the elements x16, 1 thread"
            res["tiled_sum_all"]["cpu_ms"] = round(_cpu_time(lambda: a.sum()) * 16, 1)
            res["tiled_sum_all"]["cpu_note"] = "numpy sum on 1/16 of the elements x16, 1 thread"
        del A, B, C, M, Cm

    if want("rng"):
        # Host-level Philox2x32-7 fills (src/language/random.jl:759-818): write-only streams.
        from cutile_jl_amd import random as R
        n = 1 << 27
        out = torch.empty(n, device="cuda")
        rng = R.RNG(42)
        for key, name, fn in (("rng_rand_f32", "Random.rand!(RNG, A), 2^27 f32", lambda: R.rand_(rng, out)),
                              ("rng_randn_f32", "Random.randn!(RNG, A), 2^27 f32 (Box-Muller)", lambda: R.randn_(rng, out))):
            res[key] = _entry(name, fn, 4 * n, "GB/s", "hbm", HBM_PEAK_GBS, "u32" if "rand_f32" in key else "f32", nruns, warmup)
            res[key]["variant"] = ct.last_variant()
        if cpu:
            g = np.random.Generator(np.random.Philox(42))
            res["rng_rand_f32"]["cpu_ms"] = round(_cpu_time(lambda: g.random(n // 16, dtype=np.float32)) * 16, 1)
            res["rng_rand_f32"]["cpu_note"] = "numpy Generator(Philox) float32 uniforms, 1/16 of the elements x16, 1 thread"
        del out

    if want("moe"):
        d = moe.prepare(benchmark=True, topk=2, router="top2_logits")
        flop = moe.metric(d)[0]
        wbytes = (d.w1.numel() + d.w2.numel()) * 2 + 2 * d.hidden_states.numel() * 2
        tok, exp = ct.moe_align_tile_size(d.topk_ids.cpu(), 128, d.num_experts)
        al = (tok.cuda(), exp.cuda())

        def graph_of(fn):
            """Replayable HIP graph of the device work."""
            s = torch.cuda.Stream()
            s.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(s):
                fn()
            torch.cuda.current_stream().wait_stream(s)
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                outv = fn()
            return g, outv

        def extra(e):
            e["flop"] = flop
            e["tflops"] = round(flop / (e["avg_ms"] * 1e-3) / 1e12, 2)
            e["mfma_frac"] = round(e["tflops"] / 2500.0, 5)
            return e

        whole = lambda: moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 128, 128, 64,
                                       device_align=False, fuse_silu=False)   # the reference's orchestration, moe.jl:218-257
        res["moe_f16"] = extra(_entry("MoE f16 256tok/1024h/32e/2048i top-2, cutile_moe as the reference orchestrates it (host sort + H2D/D2H inside, 4 kernels)",
                                      whole, wbytes, "GB/s", "hbm", HBM_PEAK_GBS, "f16", nruns, warmup))
        whole_dev = lambda: moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 128, 128, 64,
                                           device_align=True, fuse_silu=False, fuse_sum=False)
        default_call = lambda: moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 128, 128, 64)
        res["moe_f16_default"] = extra(_entry("MoE f16 top-2, cutile_moe with its defaults (token sort on the GPU, SiLU*up fused, down projection adding into the output: 3 launches; eager, incl. allocations)",
                                              default_call, wbytes, "GB/s", "hbm", HBM_PEAK_GBS, "f16", nruns, warmup))
        res["moe_f16_device_align"] = extra(_entry("MoE f16 top-2, whole cutile_moe with the token sort on the GPU (no host round trip; eager launches)",
                                                   whole_dev, wbytes, "GB/s", "hbm", HBM_PEAK_GBS, "f16", nruns, warmup))
        dev = whole_dev
        ref_out = dev()
        try:
            g, gout = graph_of(dev)
            g.replay(); torch.cuda.synchronize()
            assert torch.equal(gout, ref_out), "graph replay differs from eager"
            res["moe_f16_device"] = extra(_entry("MoE f16 top-2, whole cutile_moe on the device (token sort + 4 kernels), HIP graph replay",
                                                 g.replay, wbytes, "GB/s", "hbm", HBM_PEAK_GBS, "f16", nruns, warmup))
        except Exception as ex:  # graph capture unavailable: fall back to eager launches
            res["moe_f16_device"] = extra(_entry(f"MoE f16 top-2, device work only (eager; graph failed: {type(ex).__name__})",
                                                 dev, wbytes, "GB/s", "hbm", HBM_PEAK_GBS, "f16", nruns, warmup))
        fused = lambda: moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 128, 128, 64,
                                       device_align=True, fuse_silu=True)
        assert torch.equal(fused(), ref_out), "fused SiLU epilogue differs from the separate kernels"
        try:
            gf, _ = graph_of(fused)
            res["moe_f16_device_fused"] = extra(_entry("MoE f16 top-2 on the device, SiLU*up fused into the gate/up GEMM epilogue and the top-k sum into the down GEMM (sort + 2 GEMMs), HIP graph replay",
                                                       gf.replay, wbytes, "GB/s", "hbm", HBM_PEAK_GBS, "f16", nruns, warmup))
        except Exception as ex:
            res["moe_f16_device_fused"] = extra(_entry(f"MoE f16 top-2, fused SiLU epilogue (eager; graph failed: {type(ex).__name__})",
                                                       fused, wbytes, "GB/s", "hbm", HBM_PEAK_GBS, "f16", nruns, warmup))
        # from router logits to output without a host step: router + sort + 2 GEMMs
        logits_jl = d.logits.t().contiguous()
        rw = torch.empty_like(d.topk_weights)
        rid = torch.empty_like(d.topk_ids)

        def routed():
            ct.moe_route_topk(logits_jl, 2, topk_weights=rw, topk_ids=rid)
            return moe.cutile_moe(d.hidden_states, d.w1, d.w2, rw, rid, 128, 128, 64, device_align=True, fuse_silu=True)
        routed()
        assert torch.equal(rid, d.topk_ids), "device router picks other experts than the host router"
        try:
            gr, _ = graph_of(routed)
            res["moe_f16_device_routed"] = extra(_entry("MoE f16 top-2 from router logits to output on the device (router + sort + 2 GEMMs), HIP graph replay",
                                                        gr.replay, wbytes, "GB/s", "hbm", HBM_PEAK_GBS, "f16", nruns, warmup))
        except Exception as ex:
            res["moe_f16_device_routed"] = extra(_entry(f"MoE f16 top-2 from router logits (eager; graph failed: {type(ex).__name__})",
                                                        routed, wbytes, "GB/s", "hbm", HBM_PEAK_GBS, "f16", nruns, warmup))
        # the reference example's own routing (moe.jl:311-344: top-8 of 32 experts, 64 tokens per expert on average)
        d8 = moe.prepare(benchmark=True, topk=8)
        flop8 = moe.metric(d8)[0]
        top8 = lambda: moe.cutile_moe(d8.hidden_states, d8.w1, d8.w2, d8.topk_weights, d8.topk_ids, 128, 128, 64,
                                      device_align=True, fuse_silu=True)
        top8()
        try:
            g8k, _ = graph_of(top8)
            e8 = _entry("MoE f16 top-8 (the reference example's routing) on the device, fused SiLU epilogue, HIP graph replay",
                        g8k.replay, wbytes, "GB/s", "hbm", HBM_PEAK_GBS, "f16", nruns, warmup)
        except Exception as ex:
            e8 = _entry(f"MoE f16 top-8 on the device (eager; graph failed: {type(ex).__name__})", top8, wbytes, "GB/s", "hbm",
                        HBM_PEAK_GBS, "f16", nruns, warmup)
        e8["flop"] = flop8
        e8["tflops"] = round(flop8 / (e8["avg_ms"] * 1e-3) / 1e12, 2)
        e8["mfma_frac"] = round(e8["tflops"] / 2500.0, 5)
        res["moe_f16_top8_device_fused"] = e8
        e8["variant"] = ct.last_variant()
        del d8
        # prefill: the same layer with 4096 tokens (top-2), where the call is bound by the matrix cores and the grouped
        # GEMM for dense routing (128-slot tiles on a ring of LDS stages) does the two projections; eager launches
        dp = moe.prepare(num_tokens=4096, hidden_size=1024, num_experts=32, intermediate_size=2048, topk=2, router="top2_logits")
        flopp = moe.metric(dp)[0]
        pbytes = (dp.w1.numel() + dp.w2.numel()) * 2 + 2 * dp.hidden_states.numel() * 2
        pre = lambda: moe.cutile_moe(dp.hidden_states, dp.w1, dp.w2, dp.topk_weights, dp.topk_ids, 128, 128, 64)
        pre()
        ep = _entry("MoE f16 prefill: 4096 tokens top-2 of 32 experts, cutile_moe with its defaults (sort + 2 grouped GEMMs, eager)",
                    pre, pbytes, "GB/s", "hbm", HBM_PEAK_GBS, "f16", nruns, warmup)
        ep["variant"] = ct.last_variant()
        ep["flop"] = flopp
        ep["tflops"] = round(flopp / (ep["avg_ms"] * 1e-3) / 1e12, 2)
        ep["mfma_frac"] = round(ep["tflops"] / 2500.0, 5)
        res["moe_f16_prefill"] = ep
        # the same prefill batch with E4M3FN weights and activations: fp8 x fp8 on the matrix cores in both projections
        # (activations quantised per tensor by the library between them: sort + quantise + GEMM + quantise + GEMM)
        qp = moe.quantize_weights(dp)
        pre8 = lambda: moe.cutile_moe(dp.hidden_states, qp.w1, qp.w2, dp.topk_weights, dp.topk_ids, 128, 128, 64,
                                      w1_scale=qp.w1_scale, w2_scale=qp.w2_scale, fp8_activations=True)
        pre8()
        p8bytes = qp.w1.numel() + qp.w2.numel() + 2 * dp.hidden_states.numel() * 2
        e8p = _entry("MoE e4m3 x e4m3 prefill: 4096 tokens top-2 of 32 experts, fp8 activations and weights in both grouped GEMMs (eager)",
                     pre8, p8bytes, "GB/s", "hbm", HBM_PEAK_GBS, "fp8", nruns, warmup)
        e8p["variant"] = ct.last_variant()
        e8p["flop"] = flopp
        e8p["tflops"] = round(flopp / (e8p["avg_ms"] * 1e-3) / 1e12, 2)
        e8p["mfma_frac"] = round(e8p["tflops"] / 5000.0, 5)
        e8p["mfma_peak_used"] = "fp8 dense, 5000 TFLOP/s"
        res["moe_fp8_prefill"] = e8p
        del dp, qp
        if cpu:
            J = orc.to_julia
            args = (J(d.hidden_states), J(d.w1), J(d.w2), J(d.topk_weights), J(d.topk_ids))
            res["moe_f16"]["cpu_ms"] = round(_cpu_time(lambda: orc.ref_moe(*args), repeats=1), 1)
            res["moe_f16"]["cpu_note"] = f"numpy restatement of ref_moe, BLAS {ncores} threads"
        # fp8 weights (per-channel fp32 scales)
        q = moe.quantize_weights(d)
        w1q, w2q, s1t, s2t = q.w1, q.w2, q.w1_scale, q.w2_scale
        w8bytes = w1q.numel() + w2q.numel() + (s1t.numel() + s2t.numel()) * 4 + 2 * d.hidden_states.numel() * 2
        dev8 = lambda: moe.cutile_moe(d.hidden_states, w1q, w2q, d.topk_weights, d.topk_ids, 128, 128, 64, w1_scale=s1t,
                                      w2_scale=s2t, device_align=True, fuse_silu=True)
        dev8()
        # two more copies of the e4m3 weights (201 MB each): cycling over three sets touches 400 MB between two
        # uses of a set, more than the 256 MB memory-side cache keeps
        copies = [(w1q, w2q)] + [(w1q.clone(), w2q.clone()) for _ in range(2)]
        cold8 = [(lambda a=a, b=b: moe.cutile_moe(d.hidden_states, a, b, d.topk_weights, d.topk_ids, 128, 128, 64, w1_scale=s1t,
                                                  w2_scale=s2t, device_align=True, fuse_silu=True)) for a, b in copies]
        try:
            g8, _ = graph_of(dev8)
            gcold = [graph_of(f)[0].replay for f in cold8]
            res["moe_fp8_device"] = extra(_entry("MoE e4m3 weights top-2, whole cutile_moe on the device (fused SiLU epilogue), HIP graph replay", g8.replay,
                                                 w8bytes, "GB/s", "hbm", HBM_PEAK_GBS, "fp8 weights / f16 MFMA", nruns, warmup, cold=gcold))
        except Exception as ex:
            res["moe_fp8_device"] = extra(_entry(f"MoE e4m3 weights top-2, device work only (eager; {type(ex).__name__})", dev8,
                                                 w8bytes, "GB/s", "hbm", HBM_PEAK_GBS, "fp8 weights / f16 MFMA", nruns, warmup, cold=cold8))
        del copies, cold8
        del d
    torch.cuda.synchronize()
    return res


def parity_errors(ct):
    """Achieved error of every benchmark configuration against the float64 oracle, on the same seeded inputs
    the timing legs use (bounded samples where the CPU side would otherwise take minutes).  Per
    configuration: max_abs; max_rel_scale = max|err| / max|ref|; max_rel_elem = max |err| / |ref| over the
    elements with |ref| >= 1e-3 max|ref|; the tolerance the configuration states and whether it holds in
    the form the tests use, |err| <= tol * (|ref| + max|ref|)."""
    import numpy as np
    import torch
    from oracle import cutile_oracle as orc
    from cutile_jl_amd.examples import vadd, layernorm, softmax, matmul, batchmatmul, fmha, moe
    J = orc.to_julia
    out = {}

    def rec(name, got, ref, tol, sample):
        got = np.asarray(got, dtype=np.float64); ref = np.asarray(ref, dtype=np.float64)
        err = np.abs(got - ref)
        scale = float(np.abs(ref).max())
        big = np.abs(ref) >= 1e-3 * scale
        out[name] = {"max_abs": float(err.max()), "max_rel_scale": float(err.max() / scale) if scale else 0.0,
                     "max_rel_elem": float((err[big] / np.abs(ref[big])).max()) if big.any() else 0.0,
                     "tol": tol, "pass": bool(np.all(err <= tol * (np.abs(ref) + scale))) if tol else bool(err.max() == 0.0),
                     "sample": sample}

    d = vadd.prepare(benchmark=True)
    r = vadd.run(d)
    n = 1 << 24
    rec("vadd 2^27 f32 (bit-exact)", r.c[:n].cpu().numpy(), d.a[:n].cpu().numpy() + d.b[:n].cpu().numpy(), 0.0, "first 2^24 elements")
    del d, r
    d = layernorm.prepare(benchmark=True)
    r = layernorm.run(d)
    X, W, B, DY = J(d.X), J(d.W), J(d.B), J(d.DY)
    Y, mean, rstd = orc.layer_norm_fwd(X, W, B, d.eps)
    rec("LayerNorm fwd y", J(r.Y), Y, 1e-5, "all 4096 rows")
    del Y
    DX, DW, DB = orc.layer_norm_bwd(X, W, DY, d.eps)
    rec("LayerNorm bwd dx", J(r.DX), DX, 1e-5, "all 4096 rows")
    rec("LayerNorm bwd dgamma", J(r.FINAL_DW), DW, 1e-5, "all 4096 channels")
    rec("LayerNorm bwd dbeta", J(r.FINAL_DB), DB, 1e-5, "all 4096 channels")
    del DX
    del d, r, X, DY
    d = softmax.prepare(benchmark=True)
    r = softmax.run(d)
    rec("softmax", J(r.output_tma)[:, :256], orc.softmax(J(d.input)[:, :256]), 1e-5, "256 of 4096 columns")
    del d, r
    d = matmul.prepare(benchmark=True, T=torch.float16, out_T=torch.float32, dist="normal64")
    r = matmul.run(d)
    A = J(d.A).astype(np.float64); Bm = J(d.B).astype(np.float64)
    rws = sorted(set([0, 1, 255, 256, 2049, 4095] + list(range(37, 4096, 61))))   # every tile row and lane position
    rec("GEMM 4096^3 f16 -> f32", J(r.C)[rws], A[rws] @ Bm, 2e-2, f"{len(rws)} of 4096 rows of C")
    del d, r, A, Bm
    d = batchmatmul.prepare(benchmark=True)
    r = batchmatmul.run(d)
    rec("batched GEMM f32", J(r.C)[:, :, 0], J(d.A)[:, :, 0].astype(np.float64) @ J(d.B)[:, :, 0].astype(np.float64), 1e-5, "batch entry 1 of 8")
    del d, r
    d = fmha.prepare(benchmark=True)
    r = fmha.run(d)
    Q, K, V = (J(t)[:, :, :, ::4] for t in (d.Q, d.K, d.V))
    rec("causal FMHA f16", J(r.out)[:, :, :, ::4], orc.ref_fmha(Q, K, V, causal=True, dtype=np.float64), 2e-2, "32 of 128 (batch, head) pairs: all heads of batches 1 and 5")
    del d, r
    d = moe.prepare(benchmark=True, topk=2, router="top2_logits")
    got = moe.cutile_moe(d.hidden_states, d.w1, d.w2, d.topk_weights, d.topk_ids, 128, 128, 64)
    rec("MoE f16 top-2", J(got), orc.ref_moe(J(d.hidden_states), J(d.w1), J(d.w2), J(d.topk_weights), J(d.topk_ids), dtype=np.float32), 2e-2, "whole output")
    q = moe.quantize_weights(d)
    got = moe.cutile_moe(d.hidden_states, q.w1, q.w2, d.topk_weights, d.topk_ids, 128, 128, 64, w1_scale=q.w1_scale, w2_scale=q.w2_scale)
    w1d = orc.e4m3fn_decode(J(q.w1.view(torch.uint8))) * J(q.w1_scale)[None]
    w2d = orc.e4m3fn_decode(J(q.w2.view(torch.uint8))) * J(q.w2_scale)[None]
    rec("MoE e4m3 weights top-2 (vs ref_moe on the dequantised weights)", J(got),
        orc.ref_moe(J(d.hidden_states), w1d, w2d, J(d.topk_weights), J(d.topk_ids), dtype=np.float32), 2e-2, "whole output")
    return out


def headline(ct, steps, warmup):
    """LayerNorm fwd+bwd and softmax on 4096x4096 fp32.  Returns seconds per step,
    per-stage average durations from events inside the timed region, and algorithmic bytes."""
    import torch
    from cutile_jl_amd.examples import layernorm, softmax
    dl = layernorm.prepare(benchmark=True)
    ds = softmax.prepare(benchmark=True)
    D = {k: ct.TileArray(getattr(dl, k)) for k in ("X", "W", "B", "Y", "Mean", "Rstd", "DY", "DX", "DW_partial",
                                                   "DB_partial", "Locks", "FINAL_DW", "FINAL_DB")}
    SI, SO = ct.TileArray(ds.input), ct.TileArray(ds.output_tma)
    G = dl.GROUP_SIZE_M

    # Pre-bound launches (arguments converted once): at ~20 us per kernel the Python side of an
    # ordinary wrapper call would be the bottleneck of the timed loop.
    ln_fwd = ct.bind("mi_layer_norm_fwd", D["X"], D["W"], D["B"], D["Y"], D["Mean"], D["Rstd"], dl.eps, 1024)
    ln_bwd_main = ct.bind("mi_layer_norm_bwd_dx_partial_dwdb", D["DX"], D["DY"], D["DW_partial"], D["DB_partial"],
                          D["X"], D["W"], D["Mean"], D["Rstd"], D["Locks"], G, 1024)
    ln_bwd_final = ct.bind("mi_layer_norm_bwd_dwdb", D["DW_partial"], D["DB_partial"], D["FINAL_DW"], D["FINAL_DB"], 32, 1024)
    sm = ct.bind("mi_softmax_tma_kernel", SO, SI, 4096, ds.M)

    def fills():  # the host code's fill! of the partials before every backward (layernorm.jl:245-246), one launch
        dl.partials.zero_()

    stages = [("layer_norm_fwd", ln_fwd), ("fills", fills), ("layer_norm_bwd_dx_partial_dwdb", ln_bwd_main),
              ("layer_norm_bwd_dwdb", ln_bwd_final), ("softmax_tma_kernel", sm)]
    for _ in range(warmup):
        for _, f in stages:
            f()
    torch.cuda.synchronize()
    # Timed region: the five launches of a step back to back, with one pair of events around the dominant
    # kernel (its launch duration for the roofline entry) in some of the steps.  Events between all stages
    # would put a marker and a dispatch gap between every two kernels of the thing being timed.
    # A pair of event records costs the stream 4-5 us (two markers with a dispatch gap each), which is 5 % of a step:
    # the pair stands around the dominant kernel in every `stride`-th step (five samples of the default timed region),
    # not in all of them.
    dom_i = 2
    stride = max(1, steps // 5)
    ev = {s: (torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)) for s in range(stride // 2, steps, stride)}
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for s in range(steps):
        for i, (_, f) in enumerate(stages):
            if i == dom_i and s in ev:
                ev[s][0].record()
                f()
                ev[s][1].record()
            else:
                f()
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    dom_ms = sum(a.elapsed_time(b) for a, b in ev.values()) / len(ev)
    # Per-stage durations: a second, untimed pass with events between all stages.
    ev2 = [[torch.cuda.Event(enable_timing=True) for _ in range(len(stages) + 1)] for _ in range(steps)]
    for s in range(steps):
        ev2[s][0].record()
        for i, (_, f) in enumerate(stages):
            f()
            ev2[s][i + 1].record()
    torch.cuda.synchronize()
    per_stage = {name: sum(ev2[s][i].elapsed_time(ev2[s][i + 1]) for s in range(steps)) / steps
                 for i, (name, _) in enumerate(stages)}
    per_stage["dominant_in_timed_region"] = dom_ms
    MN4 = dl.M * dl.N * 4
    work = {
        "layer_norm_fwd": 2 * MN4 + (2 * dl.N + 2 * dl.M) * 4,
        "layer_norm_bwd_dx_partial_dwdb": 3 * MN4 + (dl.N + 2 * dl.M) * 4 + 2 * dl.N * G * 4,
        "layer_norm_bwd_dwdb": 2 * dl.N * G * 4 + 2 * dl.N * 4,
        "softmax_tma_kernel": 2 * MN4,
        "fills": 0,
    }
    return (t1 - t0) / steps, per_stage, work


def cpu_baseline_headline(sample_rows=4096):
    """numpy restatement of the reference's CPU path (Julia Base broadcast + reductions,
    examples/layernorm.jl:284-313 and softmax.jl:175-188) on `sample_rows` of the 4096 rows,
    single-threaded as Julia's broadcasting is.  GB/s on the same per-row byte count."""
    import numpy as np
    from oracle import cutile_oracle as orc
    rng = np.random.default_rng(1)
    N, M = 4096, sample_rows
    X = np.asfortranarray(rng.standard_normal((N, M), dtype=np.float32))
    W = rng.standard_normal(N, dtype=np.float32); B = rng.standard_normal(N, dtype=np.float32)
    DY = np.asfortranarray(rng.standard_normal((N, M), dtype=np.float32))
    S = np.asfortranarray(rng.standard_normal((N, M), dtype=np.float32) * 2)
    best = float("inf")
    for _ in range(5):
        t0 = time.perf_counter()
        orc.layer_norm_fwd(X, W, B, 1e-5, dtype=np.float32)
        orc.layer_norm_bwd(X, W, DY, 1e-5, dtype=np.float32)
        orc.softmax(S, dtype=np.float32)
        best = min(best, time.perf_counter() - t0)
    MN4 = M * N * 4
    work = (2 * MN4) + (3 * MN4) + (2 * MN4)
    return {"value": round(work / best / 1e9, 3), "unit": "GB/s", "cores": 1, "kind": "port",
            "sample": f"{sample_rows} of 4096 rows (N=4096 f32) of LayerNorm fwd+bwd and softmax, numpy restatement of the "
                      "examples' verify() formulas, single-threaded, min of 5 passes"}


def _measured_traffic(kernel):
    """HBM bytes per launch of ``kernel`` from the counter runs recorded under profiles/ (FETCH_SIZE and
    WRITE_SIZE, scaled as stated there), with the commit they were measured at; (None, None) if absent."""
    path = os.path.join(ROOT, "profiles", "headline_kernel_hbm_traffic.txt")
    try:
        kv = dict(line.split(":", 1) for line in open(path) if ":" in line and not line.startswith("#"))
        if kernel not in kv.get("kernel", ""):
            return None, None
        return int(kv["traffic_bytes_per_launch"].strip()), kv.get("measured_at_commit", "").strip() or None
    except Exception:
        return None, None


def _host_info():
    model = None
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except Exception:
        pass
    return {"nproc": os.cpu_count(), "cpu_model": model,
            "OPENBLAS_NUM_THREADS": os.environ.get("OPENBLAS_NUM_THREADS"), "OMP_NUM_THREADS": os.environ.get("OMP_NUM_THREADS")}


# north_star targets: (key in the per-kernel results, figure, target fraction)
TARGETS = [("vadd", "frac", 0.75), ("layernorm_fwd", "frac_cold", 0.75), ("softmax_tma", "frac_cold", 0.75),
           ("matmul", "frac", 0.60), ("fmha", "frac", 0.40), ("moe_f16_default", "mfma_frac", 0.40)]
REPORTED = [("copy_ref", "frac_cold"), ("copy_ref_runtime", "frac_cold"), ("transpose", "frac"), ("layernorm_bwd", "frac_cold"), ("layernorm_bwd_static", "frac_cold"),
            ("batchmatmul", "frac"), ("matmul_fp8", "frac"), ("moe_f16_default", "frac"), ("moe_f16_top8_device_fused", "frac"), ("moe_f16_top8_device_fused", "mfma_frac"), ("moe_f16_prefill", "mfma_frac"), ("moe_fp8_prefill", "mfma_frac"),
            ("moe_fp8_device", "frac_cold"), ("fmha_decode", "frac"), ("fmha_decode_16k", "frac")]
MAX_LINE_BYTES = 4096   # the last stdout line must stay a small record: a consumer that keeps only the end of stdout still parses it


def _summary(kernels):
    """One compact entry per north_star target (and per reported figure without a target):
    ``frac`` = fraction of the roofline from the back-to-back average (for ``*.frac_cold`` keys: while rotating
    buffer sets); ``ref`` = the same fraction from the minimum of single event-bracketed launches, the reference's
    own protocol (examples/benchmarks.jl:12-13,158-171); ``t`` = target or null; ``ok`` = target met."""
    out = {}
    for key, fig, target in TARGETS + [(k, f, None) for k, f in REPORTED]:
        e = kernels.get(key)
        if not e or fig not in e:
            continue
        rec = {"frac": e[fig]}
        if e.get("min_ms"):
            if fig == "mfma_frac":
                rec["ref"] = round(e["flop"] / (e["min_ms"] * 1e-3) / 1e12 / (5000.0 if e.get("dtype") == "fp8" else 2500.0), 4)
            else:
                scale = 1e9 if e["unit"] == "GB/s" else 1e12
                rec["ref"] = round(e["work"] / (e["min_ms"] * 1e-3) / scale / e["peak"], 4)
        if target is not None:
            rec["t"] = target
            rec["ok"] = bool(e[fig] >= target)
        out[f"{key}.{fig}"] = rec
    return out


def headline_record(full):
    """The last stdout line: the contract keys, the roofline and CPU baseline objects and the compact summary;
    everything else (per-kernel entries, achieved errors, per-stage times) stays in the full record."""
    keep = ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling",
            "vs_baseline", "dtype", "data", "config", "roofline", "cpu_baseline")
    rec = {k: full[k] for k in keep if k in full}
    if "errors" in full:
        rec["parity"] = {"configs": len(full["errors"]), "all_within_tolerance": all(e["pass"] for e in full["errors"].values())}
    if "summary" in full:
        rec["summary"] = full["summary"]
    rec["detail"] = full.get("detail_file")
    line = json.dumps(rec, allow_nan=False, separators=(",", ":"))
    if len(line) > MAX_LINE_BYTES:   # never let the record outgrow what a consumer parses: drop the optional parts
        for k in ("summary", "parity", "detail"):
            rec.pop(k, None)
            line = json.dumps(rec, allow_nan=False, separators=(",", ":"))
            if len(line) <= MAX_LINE_BYTES:
                break
    return line


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--kernels", type=str, default="all", help="comma list for the per-kernel table, 'all' or 'none'")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--table", action="store_true", help="also print a human-readable table on stderr")
    ap.add_argument("--full", action="store_true", help="print the full record (per-kernel entries, errors, stages) as a stdout line before the last one")
    ap.add_argument("--detail-file", type=str, default=os.path.join("gpurun_out", "bench_full.json"),
                    help="where the full record is written (relative to the repository root; '' = nowhere)")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one MI355X; multi-GPU runs are not part of this build (use --gpus 1)", file=sys.stderr)
        sys.exit(2)

    import torch
    import __graft_entry__ as entry
    ct = entry.load_package()
    ct.lib()
    assert torch.cuda.is_available(), "bench.py needs a GPU"
    torch.cuda.set_device(0)

    sec_per_step, per_stage, work = headline(ct, args.steps, args.warmup)
    total_work = sum(work.values())
    dom = "layer_norm_bwd_dx_partial_dwdb"      # the longest kernel of the step (see stages_ms)
    dom_ms = per_stage["dominant_in_timed_region"]
    ach = work[dom] / (dom_ms * 1e-3) / 1e9
    traffic, traffic_commit = _measured_traffic(dom)
    out = {
        "metric": "norm/softmax GB/s (LayerNorm fwd+bwd + softmax, 4096x4096 f32); FMHA/MoE/GEMM legs in summary",
        "value": round(total_work / sec_per_step / 1e9, 2), "unit": "GB/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": round(sec_per_step * 1e3, 5), "higher_is_better": True,
        "scaling": "weak", "vs_baseline": None, "dtype": "f32", "data": "synthetic",
        "config": {"workload": "configs[1]: row LayerNorm fwd+bwd (y, dx, dgamma, dbeta) + row softmax on 4096x4096 Float32",
                   "M": 4096, "N": 4096, "eps": 1e-5, "GROUP_SIZE_M": 64, "bytes_per_step": total_work},
        "roofline": {"bound": "hbm", "achieved": round(ach, 2), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": round(ach / HBM_PEAK_GBS, 4),
                     # HBM bytes per launch from the rocprofv3 FETCH_SIZE / WRITE_SIZE runs recorded in
                     # profiles/headline_kernel_hbm_traffic.txt (null if that record is absent)
                     "traffic": traffic, "kernel": dom,
                     "avg_launch_ms": round(dom_ms, 5), "algorithmic_bytes": work[dom]},
        "traffic_measured_at_commit": traffic_commit,
        "seeds": {"layernorm": 1, "softmax": 2, "matmul": 3, "batchmatmul": 4, "fmha": 5, "moe": 6, "vadd": 0},
        "stages_ms": {k: round(v, 5) for k, v in per_stage.items()},
        "stages_frac": {k: round(work[k] / (per_stage[k] * 1e-3) / 1e9 / HBM_PEAK_GBS, 4) for k in work if work[k]},
        "shader_clock_mhz_idle": _shader_clock_mhz(),
    }
    if not args.no_cpu:
        out["cpu_baseline"] = cpu_baseline_headline()
        out["host"] = _host_info()
        out["errors"] = parity_errors(ct)
    if args.kernels != "none":
        which = None if args.kernels == "all" else set(args.kernels.split(","))
        out["kernels"] = bench_kernels(ct, which, cpu=not args.no_cpu)
    if args.table and "kernels" in out:
        flat = [r for e in out["kernels"].values() for r in e.get("rows", [e])]
        for e in flat:
            cpu = f"  cpu {e['cpu_ms']:10.1f} ms" if "cpu_ms" in e else ""
            cold = f"  cold {100 * e['frac_cold']:6.2f}%" if "frac_cold" in e else ""
            print(f"{e['name'][:72]:<72} min {e['min_ms']:8.4f}  avg {e['avg_ms']:8.4f} ms  "
                  f"{e['achieved']:9.1f} {e['unit']:<8} {100 * e['frac']:6.2f}% of {e['bound']} peak{cold}{cpu}", file=sys.stderr)
    if "kernels" in out:
        out["summary"] = _summary(out["kernels"])
    if args.detail_file:
        path = os.path.join(ROOT, args.detail_file)
        try:
            os.makedirs(os.path.dirname(path), exist_ok=True)
            with open(path, "w") as f:
                json.dump(out, f, indent=1)
            out["detail_file"] = args.detail_file
        except OSError as ex:
            print(f"bench.py: could not write {path}: {ex}", file=sys.stderr)
    if args.full:
        print(json.dumps(out))
    sys.stdout.flush()
    print(headline_record(out))


if __name__ == "__main__":
    main()
