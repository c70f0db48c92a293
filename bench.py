#!/usr/bin/env python3
"""Benchmark of the SGEMM hot path on one MI355X (gfx950).

Headline workload: SGEMM M = N = K = 8192, row-major NN, alpha = 1.5,
beta = 0.5, A, B, C ~ U[-1, 1) (24-bit, seeded), inputs resident in HBM.
A "step" is one call of the headline form: the fastest form whose max and
mean relative error vs FP64 are no worse than the plain FP32 kernel's -- the
2-way fp16 split with per-row power-of-two scales (FP16X3) on MFMA.  The
plain FP32 kernel and the other forms (BF16x3, FP32 on the FP32 matrix
cores, BF16x6, BF16x1, FP8 block-scaled) are timed the same way beside it,
each with its error ratios.  Timing: W untimed warm-up calls, then K
calls bracketed by device synchronisation and HIP events on the launch stream.
The dominant kernel's own average duration (the MFMA core, without the
operand-preparation kernels) comes from the library's event hook
(ugemm_hip_timing_*), recorded on the same stream.

Also reported (one JSON line in total, with the main figures; all of them in
the [detail] line on stderr):
  * errors of every form vs an FP64 evaluation of 64 sampled rows;
  * config 2's grid: 2048^3, 4096^3, 8192^3 x NN/NT/TN for FP32, BF16x3 and
    FP16X3, each cell with its roofline fraction and errors;
  * tall-skinny / short-wide SGEMM and the 4096^3 DGEMM (normal(0,1) inputs,
    DGEMM bit-compared across two runs);
  * 512 uneven im2col-shaped problems on independent operands (6.9 GB
    resident) in one grouped persistent launch (hipGraph replay) per form,
    every problem checked on 2 sampled rows, vs a loop of plain-kernel
    launches; a cache-resident pooled-operand variant as a labelled extra;
    and the same 512
    shapes as 3x3 convolutions with implicit im2col and the bias + LeakyReLU
    epilogue;
  * the precision ladder at 8192^3 with entries sign * 2^e * (1+u), e in [-12, 12];
  * the BLAS-1/2 helpers (axpy, gemv) against the HBM roofline;
  * host-pointer calls with copies included (sgemm_test.c's workload, and
    one 8192^3 uut call);
  * cpu_baseline: the reference's own sgemm_avx (compiled from its sources
    into oracle/_ref) on a bounded row band of the 8192^3 workload, one thread;
    beside it the same on every host core, dgemm_avx on one thread, and
    (full run) config 1: sgemm_avx and sgemm_c at 1024^3 against FP64.
"""
import argparse
import json
import os
import platform
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

import ugemm_amd as ug  # noqa: E402
from ugemm_amd import hip  # noqa: E402

# MI355X published dense peaks (TFLOP/s) and HBM bandwidth.
PEAK = {"fp32_vector": 157.3, "fp32_mfma": 157.3, "bf16_mfma": 2516.6, "fp16_mfma": 2516.6, "fp8_mfma": 5033.2, "fp64": 78.6}
HBM_GBPS = 8000.0
# Form -> (peak used for roofline.frac, MFMA products per useful product)
FORM_PEAK = {"fp32": ("fp32_vector", 1), "bf16x3": ("bf16_mfma", 3), "bf16x6": ("bf16_mfma", 6),
             "fp16x3": ("fp16_mfma", 3), "fp32_mfma": ("fp32_mfma", 1),
             "bf16x1": ("bf16_mfma", 1), "fp8": ("fp8_mfma", 1)}
# Arithmetic each form computes in (the bench line's dtype).
DTYPE = {"fp32": "f32 (vector FMA)", "fp32_mfma": "f32 (FP32 MFMA, f32 accumulate)",
         "fp16x3": "f32 via a 2-way fp16 split with per-row power-of-two scales on MFMA, f32 accumulate",
         "bf16x3": "f32 via a 2-way bf16 split on MFMA, f32 accumulate",
         "bf16x6": "f32 via a 3-way bf16 split on MFMA, f32 accumulate",
         "bf16x1": "bf16 operands on MFMA, f32 accumulate", "fp8": "fp8-e4m3 with 128x128 block scales, f32 accumulate"}
CORE_KERNEL = {"fp32": "sgemm_fp32_kernel", "bf16x3": "split_nt_core", "bf16x6": "split_nt_core",
               "fp16x3": "split_nt_core", "fp32_mfma": "sgemm_mfma32_kernel",
               "bf16x1": "split_nt_core", "fp8": "fp8_scaled_core"}


def log(*a):
    print(*a, file=sys.stderr, flush=True)


def uniform(g, shape):
    k = g.integers(0, 1 << 24, size=shape, dtype=np.int64)
    return (k.astype(np.float32) * np.float32(2.0 ** -23) - np.float32(1.0))


def wide(g, shape):
    s = np.where(g.integers(0, 2, size=shape) == 0, -1.0, 1.0)
    e = g.integers(-12, 13, size=shape)
    u = g.integers(0, 1 << 23, size=shape).astype(np.float64) * 2.0 ** -23
    return (s * np.ldexp(1.0 + u, e)).astype(np.float32)


LAST_STEPS = {}   # per-step median and minimum of the last timed() call


def timed(fn, steps, warmup, stream, warm_ms=0.0):
    """(ms per step from events, ms per core kernel launch, wall seconds of
    the timed steps).  The core time, and the per-step median and minimum in
    LAST_STEPS, come from a second, instrumented pass over as many steps.

    `warmup` untimed calls, then (warm_ms > 0) more untimed calls until
    warm_ms of wall time has passed: the GPU's clock rises over the first
    ~100 ms of sustained load after an idle spell (host-side work between
    sections), and a few calls do not reach it (measured: a 0.5 ms GEMM
    timed right after an idle spell ran 20% slower than the same GEMM
    0.3 s later)."""
    t_w = time.perf_counter()
    for _ in range(warmup):
        fn()
    stream.synchronize()
    while warm_ms > 0 and (time.perf_counter() - t_w) * 1e3 < warm_ms:
        for _ in range(4):
            fn()
        stream.synchronize()
    hip.synchronize()
    # The timed steps: one event before the first and one after the last,
    # nothing else on the stream (each event recorded between steps, and the
    # library's own core-kernel events, add 5-12 us of gaps per step:
    # measured 79 against 67 us per 2048^3 BF16x3 call).
    e0, e1 = hip.Event(), hip.Event()
    t0 = time.perf_counter()
    e0.record(stream)
    for _ in range(steps):
        fn()
    e1.record(stream)
    e1.synchronize()
    hip.synchronize()
    wall = time.perf_counter() - t0
    ms = e0.elapsed_ms(e1) / steps
    e0.destroy()
    e1.destroy()
    # Then the same steps again, instrumented: an event between consecutive
    # steps (per-step median and minimum) and the core kernel's own launch
    # time, from events the library records around it.
    ev = [hip.Event() for _ in range(steps + 1)]
    ug.timing_enable(True)
    ev[0].record(stream)
    for i in range(steps):
        fn()
        ev[i + 1].record(stream)
    ev[-1].synchronize()
    hip.synchronize()
    n, core_ms = ug.timing_collect()
    ug.timing_enable(False)
    per = sorted(ev[i].elapsed_ms(ev[i + 1]) for i in range(steps))
    LAST_STEPS["median_ms"], LAST_STEPS["min_ms"] = per[len(per) // 2], per[0]
    for e in ev:
        e.destroy()
    return ms, (core_ms / n if n else None), wall


def mfma_sustained(rounds=20000):
    """The device's sustained 16x16x32 MFMA rate (TFLOP/s) for bf16 and f16
    operands: every SIMD issues nothing but independent MFMAs for ~25 ms
    (ugemm_hip_mfma_ceiling), the rate any split-form core can reach under the
    power limit.  The operands are planes of the headline's data: U[-1,1)
    split into hi + lo (bf16, round to nearest even; fp16 after the 2^15 row
    scale FP16X3 applies), since the rate depends on the bits multiplied."""
    g = np.random.Generator(np.random.PCG64(0x55474D4D0C))
    x = uniform(g, 4096).astype(np.float32)
    u = x.view(np.uint32)
    hi = ((u + np.uint32(0x7FFF) + ((u >> 16) & 1)) & np.uint32(0xFFFF0000)).view(np.float32)
    r = (x - hi).view(np.uint32)
    lo = ((r + np.uint32(0x7FFF) + ((r >> 16) & 1)) & np.uint32(0xFFFF0000))
    bf = np.concatenate([(hi.view(np.uint32) >> 16), lo >> 16]).astype(np.uint16)
    xs = x * np.float32(32768.0)
    h16 = xs.astype(np.float16)
    f16 = np.concatenate([h16, (xs - h16.astype(np.float32)).astype(np.float16)]).view(np.uint16)
    out = {}
    for name, planes, fp16 in (("bf16", bf, False), ("f16", f16, True)):
        d = hip.DeviceArray.from_host(planes)
        out[name] = round(max(ug.mfma_ceiling(d.ptr, fp16, rounds) for _ in range(2)), 1)
        d.free()
    return out


def warm(fn, stream, ms=250.0):
    """Untimed calls of fn until ms of wall time has passed (see timed)."""
    t0 = time.perf_counter()
    while (time.perf_counter() - t0) * 1e3 < ms:
        fn()
        stream.synchronize()


def err_stats(got, exact, scale):
    got = got.astype(np.float64)
    d = np.abs(got - exact)
    nz = exact != 0
    rel = d[nz] / np.abs(exact[nz])
    with np.errstate(divide="ignore", invalid="ignore"):
        bn = np.where(scale > 0, d / scale, 0.0)
    return {"max_rel_err": float(rel.max()), "mean_rel_err": float(rel.mean()),
            "max_abs_err": float(d.max()), "rms_abs_err": float(np.sqrt(np.mean(d * d))),
            "max_err_over_bound_scale": float(bn.max())}


def sgemm_forms(n, A, B, C0, alpha, beta, forms, steps, warmup, stream, rows, tag, headline=None):
    dA, dB, dC = hip.DeviceArray.from_host(A), hip.DeviceArray.from_host(B), hip.DeviceArray.from_host(C0)
    A64 = A[rows].astype(np.float64)
    B64 = B.astype(np.float64)
    exact = alpha * (A64 @ B64) + beta * C0[rows].astype(np.float64)
    scale = abs(alpha) * (np.abs(A64) @ np.abs(B64)) + abs(beta) * np.abs(C0[rows].astype(np.float64))
    del B64
    flop = 2.0 * n ** 3
    out = {}
    for name in forms:
        mid = ug.MODES[name]

        def call():
            ug.sgemm_dev("R", "N", "N", n, n, n, alpha, dA, n, dB, n, beta, dC, n, mode=mid, stream=stream)
        try:
            # The headline form gets exactly `warmup` untimed calls (the bench
            # contract); every other line is also warmed for 250 ms.
            ms, core_ms, wall = timed(call, steps, warmup, stream, 0.0 if name == headline else 250.0)
        except ug.UgemmError as e:
            out[name] = {"error": str(e)}
            continue
        dC.upload(C0)
        call()
        stream.synchronize()
        got = dC.download()[rows]
        peak_key, mult = FORM_PEAK[name]
        tf = flop / (ms * 1e-3) / 1e12
        rec = {"tflops": round(tf, 3), "ms_per_call": round(ms, 4), "ms_median": round(LAST_STEPS["median_ms"], 4),
               "ms_min": round(LAST_STEPS["min_ms"], 4), "wall_s": round(wall, 3),
               "core_kernel": CORE_KERNEL[name], "core_ms": round(core_ms, 4) if core_ms else None,
               "core_tflops": round(flop / (core_ms * 1e-3) / 1e12, 3) if core_ms else None,
               "frac_of_fp32_vector_peak": round(tf / PEAK["fp32_vector"], 4),
               "mfma_utilisation": round(tf * mult / PEAK[peak_key], 4) if name != "fp32" else None}
        rec.update(err_stats(got, exact, scale))
        out[name] = rec
        log(f"[{tag}] {name}: {tf:.1f} TFLOP/s ({ms:.3f} ms/call, core {core_ms:.3f} ms), "
            f"max rel err {rec['max_rel_err']:.3g}, rms abs {rec['rms_abs_err']:.3g}")
    for d in (dA, dB, dC):
        d.free()
    return out


def config2_grid(stream, steps, sizes=(2048, 4096, 8192), layouts=("NN", "NT", "TN"),
                 forms=("fp32", "bf16x3", "fp16x3")):
    """Config 2's grid: M = N = K in `sizes`, row-major layouts NN/NT/TN (the
    RNN/RNT/RTN cases sgemm_test.c:229-263 times), alpha = 1.5, beta = 0.5,
    A, B, C ~ U[-1, 1) (24-bit, seed 0x55474D4D02 + n).  Per cell: TFLOP/s per
    call (operand preparation included), the core kernel's rate, the fraction
    of the form's roofline (FP32 vector peak for fp32; the MFMA peak at
    algorithmic flops for the split forms, with the issued-MFMA fraction), and
    max/mean relative error vs FP64 on 32 sampled rows."""
    alpha, beta = 1.5, 0.5
    res = {}
    for n in sizes:
        g = np.random.Generator(np.random.PCG64(0x55474D4D02 + n))
        A, B, C0 = uniform(g, (n, n)), uniform(g, (n, n)), uniform(g, (n, n))
        dA, dB, dC = hip.DeviceArray.from_host(A), hip.DeviceArray.from_host(B), hip.DeviceArray.from_host(C0)
        rows = np.sort(np.random.Generator(np.random.PCG64(12)).choice(n, 32, replace=False))
        C0r = C0[rows].astype(np.float64)
        flop = 2.0 * n ** 3
        cell_steps = max(5, steps // 2) if n >= 8192 else steps
        for lay in layouts:
            ta, tb = lay[0], lay[1]
            Ar = (A[rows] if ta == "N" else A[:, rows].T).astype(np.float64)
            Bop = (B if tb == "N" else B.T).astype(np.float64)
            exact = alpha * (Ar @ Bop) + beta * C0r
            scale = abs(alpha) * (np.abs(Ar) @ np.abs(Bop)) + abs(beta) * np.abs(C0r)
            del Bop
            for form in forms:
                mid = ug.MODES[form]

                def call():
                    ug.sgemm_dev("R", ta, tb, n, n, n, alpha, dA, n, dB, n, beta, dC, n, mode=mid, stream=stream)
                ms, core_ms, _ = timed(call, cell_steps, 2, stream, 150.0)
                dC.upload(C0)
                call()
                stream.synchronize()
                got = dC.download()[rows]
                peak_key, mult = FORM_PEAK[form]
                tf = flop / (ms * 1e-3) / 1e12
                core_tf = flop / (core_ms * 1e-3) / 1e12 if core_ms else None
                rec = {"tflops": round(tf, 3), "ms_per_call": round(ms, 4),
                       "core_tflops": round(core_tf, 3) if core_tf else None,
                       "roofline_peak": PEAK[peak_key],
                       "frac_of_roofline": round((core_tf or tf) / PEAK[peak_key], 4),
                       "mfma_issue_frac": round((core_tf or tf) * mult / PEAK[peak_key], 4) if form != "fp32" else None,
                       "frac_of_fp32_vector_peak": round(tf / PEAK["fp32_vector"], 4)}
                rec.update(err_stats(got, exact, scale))
                res[f"{n}_{lay}_{form}"] = rec
                log(f"[config2] {n}^3 {lay} {form}: {tf:.1f} TFLOP/s (core {core_tf or 0:.1f}), "
                    f"max rel {rec['max_rel_err']:.3g}, mean rel {rec['mean_rel_err']:.3g}")
        for d in (dA, dB, dC):
            d.free()
    # The accuracy target per cell: the split form's max and mean relative
    # error no worse than plain FP32's on the same cell.
    for n in sizes:
        for lay in layouts:
            p = res.get(f"{n}_{lay}_fp32")
            for form in forms:
                r = res.get(f"{n}_{lay}_{form}")
                if form == "fp32" or not p or not r:
                    continue
                r["speedup_vs_fp32"] = round(r["tflops"] / p["tflops"], 3)
                r["error_no_worse_than_fp32"] = bool(r["max_rel_err"] <= p["max_rel_err"]
                                                     and r["mean_rel_err"] <= p["mean_rel_err"])
    return res


def config3(stream, steps, warmup):
    """Tall-skinny and short-wide SGEMM, DGEMM 4096^3; normal(0,1); alpha=1, beta=0."""
    g = np.random.Generator(np.random.PCG64(0x55474D4D03))
    res = {}
    big = g.standard_normal((65536, 4096), dtype=np.float32)
    small = g.standard_normal((4096, 256), dtype=np.float32)
    for (M, N, K, A, B, label) in ((65536, 256, 4096, big, small, "sgemm_65536x256x4096"),
                                   (256, 65536, 4096, small.T.copy(), big.T.copy(), "sgemm_256x65536x4096")):
        dA, dB, dC = hip.DeviceArray.from_host(A), hip.DeviceArray.from_host(B), hip.DeviceArray((M, N), np.float32)
        rows = np.sort(np.random.Generator(np.random.PCG64(4)).choice(M, 32, replace=False))
        exact = A[rows].astype(np.float64) @ B.astype(np.float64)
        scale = np.abs(A[rows].astype(np.float64)) @ np.abs(B.astype(np.float64))
        res[label] = {}
        for name in ("fp32", "fp32_mfma", "bf16x3", "fp16x3", "bf16x6"):
            mid = ug.MODES[name]

            def call():
                ug.sgemm_dev("R", "N", "N", M, N, K, 1.0, dA, K, dB, N, 0.0, dC, N, mode=mid, stream=stream)
            ms, core_ms, _ = timed(call, steps, warmup, stream, 250.0)
            got = dC.download()[rows]
            r = {"tflops": round(2.0 * M * N * K / (ms * 1e-3) / 1e12, 3), "ms_per_call": round(ms, 4)}
            r.update(err_stats(got, exact, scale))
            res[label][name] = r
            log(f"[config3] {label} {name}: {r['tflops']:.1f} TFLOP/s")
        for d in (dA, dB, dC):
            d.free()
    res["dgemm_4096"] = dgemm_4096(stream, steps, g)
    return res


def dgemm_4096(stream, steps, g=None):
    """DGEMM 4096^3 R/N/N, normal(0,1), alpha = 1, beta = 0, bit-compared across two runs."""
    g = g if g is not None else np.random.Generator(np.random.PCG64(0x55474D4D03))
    n = 4096
    A = g.standard_normal((n, n))
    B = g.standard_normal((n, n))
    dA, dB = hip.DeviceArray.from_host(A), hip.DeviceArray.from_host(B)
    dC, dC2 = hip.DeviceArray((n, n), np.float64), hip.DeviceArray((n, n), np.float64)

    def call():
        ug.dgemm_dev("R", "N", "N", n, n, n, 1.0, dA, n, dB, n, 0.0, dC, n, stream=stream)
    ms, core_ms, _ = timed(call, max(3, steps // 2), 1, stream, 250.0)
    ug.dgemm_dev("R", "N", "N", n, n, n, 1.0, dA, n, dB, n, 0.0, dC2, n, stream=stream)
    stream.synchronize()
    C1, C2 = dC.download(), dC2.download()
    rows = np.sort(np.random.Generator(np.random.PCG64(5)).choice(n, 16, replace=False))
    exact = A[rows] @ B      # FP64 BLAS; the bound below is relative to |A||B|
    scale = np.abs(A[rows]) @ np.abs(B)
    r = {"tflops": round(2.0 * n ** 3 / (ms * 1e-3) / 1e12, 3), "ms_per_call": round(ms, 4),
         "frac_of_fp64_peak": round(2.0 * n ** 3 / (ms * 1e-3) / 1e12 / PEAK["fp64"], 4),
         "bitwise_reproducible": bool(np.array_equal(C1.view(np.uint64), C2.view(np.uint64)))}
    r.update(err_stats(C1[rows], exact, scale))
    log(f"[config3] dgemm 4096^3: {r['tflops']:.1f} TFLOP/s, reproducible {r['bitwise_reproducible']}")
    for d in (dA, dB, dC, dC2):
        d.free()
    return r


def config4_shapes():
    """The 512 draws of config 4: M = 32*U{1..16}, N = H*W with H = W in
    {7, 14, 28, 56}, K = 9*16*U{1..32} (seed 0x55474D4D04)."""
    g = np.random.Generator(np.random.PCG64(0x55474D4D04))
    count = 512
    Ms = 32 * g.integers(1, 17, size=count)
    HW = g.choice([7, 14, 28, 56], size=count)
    Ks = 144 * g.integers(1, 33, size=count)
    return g, Ms, HW, Ks


def config4_operands(Ms, Ns, Ks, nrows=2):
    """Independent operands for every problem: A_i (M x K) and B_i (K x N)
    U[-1, 1) (24-bit) from their own seed 0x55474D4D0400 + i, each in its own
    256-byte aligned span of one device buffer, C_i disjoint.  Returns the
    device buffers, element offsets, and per problem `nrows` sampled rows of
    C with their FP64 values and |A||B| scales (computed while the operands
    are on the host, so nothing is regenerated for the checks)."""
    def offsets(sizes):
        sz = (np.asarray(sizes, np.int64) + 63) // 64 * 64
        return np.concatenate([[0], np.cumsum(sz)])
    a_off, b_off, c_off = offsets(Ms * Ks), offsets(Ks * Ns), offsets(Ms * Ns)
    dA, dB = hip.DeviceArray(int(a_off[-1]), np.float32), hip.DeviceArray(int(b_off[-1]), np.float32)
    dC = hip.DeviceArray(int(c_off[-1]), np.float32)

    def make(i):
        M, N, K = int(Ms[i]), int(Ns[i]), int(Ks[i])
        gi = np.random.Generator(np.random.PCG64(0x55474D4D0400 + i))
        A = gi.random((M, K), dtype=np.float32) * np.float32(2.0) - np.float32(1.0)
        B = gi.random((K, N), dtype=np.float32) * np.float32(2.0) - np.float32(1.0)
        rows = np.sort(gi.choice(M, nrows, replace=False))
        Ar, B64 = A[rows].astype(np.float64), B.astype(np.float64)
        exact = Ar @ B64
        np.abs(B64, out=B64)
        return A, B, (rows, exact, np.abs(Ar) @ B64)

    import concurrent.futures as cf
    from threadpoolctl import threadpool_limits
    checks = []
    # Each problem has its own generator; one BLAS thread per worker.
    with threadpool_limits(1), cf.ThreadPoolExecutor(8) as ex:
        for c0 in range(0, len(Ms), 32):
            for i, (A, B, chk) in zip(range(c0, len(Ms)), ex.map(make, range(c0, min(len(Ms), c0 + 32)))):
                hip.check(hip.lib().hipMemcpy(dA.at(a_off[i]), A.ctypes.data, A.nbytes, hip.H2D), "config4 A")
                hip.check(hip.lib().hipMemcpy(dB.at(b_off[i]), B.ctypes.data, B.nbytes, hip.H2D), "config4 B")
                checks.append(chk)
    resident = int(4 * (a_off[-1] + b_off[-1] + c_off[-1]))
    return dA, dB, dC, a_off, b_off, c_off, checks, resident


def config4_check(dC, c_off, Ms, Ns, Ks, checks, extra):
    """Worst |C - C64| / bound over the sampled rows of every problem
    (bound: (2(K+1)eps32 + extra) |A||B|)."""
    C = dC.download()
    worst = 0.0
    for i, (rows, exact, scale) in enumerate(checks):
        M, N, K = int(Ms[i]), int(Ns[i]), int(Ks[i])
        got = C[c_off[i]:c_off[i] + M * N].reshape(M, N)[rows].astype(np.float64)
        bound = (2 * (K + 1) * 2.0 ** -24 + extra) * scale
        worst = max(worst, float(np.max(np.abs(got - exact) / bound)))
    return worst


def time_plan(plan, stream, reps=10):
    warm(lambda: plan.run(stream), stream)
    e0, e1 = hip.Event(), hip.Event()
    e0.record(stream)
    for _ in range(reps):
        plan.run(stream)           # one graph launch per run
    e1.record(stream)
    e1.synchronize()
    ms = e0.elapsed_ms(e1) / reps
    e0.destroy()
    e1.destroy()
    return ms


def config4(stream, fp32_single_tf, single_tf_by_form=None):
    """512 uneven im2col-shaped FP32 problems (config4_shapes) on independent
    operands: one grouped persistent launch per form (FP32 vector FMA, and the
    BF16x3, FP16X3 and FP32-MFMA plans), against a loop of single calls;
    2 sampled rows of every problem checked against FP64 for every form."""
    _, Ms, HW, Ks = config4_shapes()
    Ns = HW * HW
    count = len(Ms)
    flop = float(np.sum(2.0 * Ms * Ns * Ks))
    t0 = time.perf_counter()
    dA, dB, dC, a_off, b_off, c_off, checks, resident = config4_operands(Ms, Ns, Ks)
    log(f"[config4] {count} independent problems, {resident / 1e9:.2f} GB resident "
        f"(generated and uploaded in {time.perf_counter() - t0:.1f} s)")
    probs = [ug.Problem(b"N", b"N", int(Ms[i]), int(Ns[i]), int(Ks[i]), 1.0, 0.0, dA.at(a_off[i]), int(Ks[i]),
                        dB.at(b_off[i]), int(Ns[i]), dC.at(c_off[i]), int(Ns[i])) for i in range(count)]
    legs = {}
    for form, extra in (("fp32", 0.0), ("bf16x3", 2.0 ** -14), ("fp16x3", 2.0 ** -19), ("fp32_mfma", 0.0)):
        plan = ug.GroupedPlan(probs, mode=ug.MODES[form], capture=True)
        tuned = plan.tune()
        ms = time_plan(plan, stream)
        plan.destroy()
        tf = flop / (ms * 1e-3) / 1e12
        single = fp32_single_tf if form == "fp32" else (single_tf_by_form or {}).get(form)
        legs[form] = {"variant": ug.grouped_variants(ug.MODES[form])[tuned], "grouped_graph_ms": round(ms, 4),
                      "grouped_tflops": round(tf, 3), "gemms_per_s": round(count / (ms * 1e-3), 1),
                      "frac_of_single_large_gemm_rate": round(tf / single, 4) if single else None,
                      "all_problems_2_rows_worst_err_over_bound": config4_check(dC, c_off, Ms, Ns, Ks, checks,
                                                                                 extra)}
    # Baseline: a loop of plain-kernel calls over the same problems.
    loop_reps = 3

    def loop():
        for p in probs:
            ug.sgemm_dev("R", "N", "N", p.M, p.N, p.K, 1.0, p.A, p.lda, p.B, p.ldb, 0.0, p.C, p.ldc, stream=stream)
    warm(loop, stream)
    e0, e1 = hip.Event(), hip.Event()
    e0.record(stream)
    for _ in range(loop_reps):
        loop()
    e1.record(stream)
    e1.synchronize()
    ms_loop = e0.elapsed_ms(e1) / loop_reps
    e0.destroy()
    e1.destroy()
    for d in (dA, dB, dC):
        d.free()
    fp = legs.pop("fp32")
    r = {"problems": count, "gflop": round(flop / 1e9, 2), "operands": "independent per problem",
         "resident_operand_bytes": resident, "tuned_variant": fp["variant"],
         "grouped_graph_ms": fp["grouped_graph_ms"], "grouped_tflops": fp["grouped_tflops"],
         "gemms_per_s": fp["gemms_per_s"],
         "loop_plain_ms": round(ms_loop, 4), "loop_plain_tflops": round(flop / (ms_loop * 1e-3) / 1e12, 3),
         "speedup_vs_loop": round(ms_loop / fp["grouped_graph_ms"], 3),
         "frac_of_single_large_gemm_rate": fp["frac_of_single_large_gemm_rate"],
         "all_problems_2_rows_worst_err_over_bound": fp["all_problems_2_rows_worst_err_over_bound"]}
    for k, v in legs.items():
        r[k + "_grouped"] = v
    r["pooled_operands_extra"] = config4_pooled(Ms, Ns, Ks, stream, flop, fp32_single_tf)
    log(f"[config4] grouped {fp['grouped_tflops']:.1f} TFLOP/s ({fp['grouped_graph_ms']:.3f} ms), loop "
        f"{r['loop_plain_tflops']:.1f} TFLOP/s, {r['frac_of_single_large_gemm_rate']} of single-GEMM rate; "
        + ", ".join(f"{k} {v['grouped_tflops']:.1f} ({v['frac_of_single_large_gemm_rate']})" for k, v in legs.items()))
    return r


def config4_pooled(Ms, Ns, Ks, stream, flop, fp32_single_tf):
    """A labelled extra, not config 4 as stated: the same 512 shapes with
    every A sliced from one 16 MiB pool and every B from one 64 MiB pool
    (84 MB of operands, resident in the Infinity Cache), FP32 grouped."""
    g = np.random.Generator(np.random.PCG64(0x55474D4D44))
    count = len(Ms)
    pa, pb = uniform(g, 4 << 20), uniform(g, 16 << 20)
    dpa, dpb = hip.DeviceArray.from_host(pa), hip.DeviceArray.from_host(pb)
    c_off = np.concatenate([[0], np.cumsum(((Ms * Ns + 3) // 4) * 4)])
    dC = hip.DeviceArray(int(c_off[-1]), np.float32)
    a_off = 4 * g.integers(0, ((4 << 20) - Ms * Ks) // 4)
    b_off = 4 * g.integers(0, ((16 << 20) - Ks * Ns) // 4)
    probs = [ug.Problem(b"N", b"N", int(Ms[i]), int(Ns[i]), int(Ks[i]), 1.0, 0.0, dpa.at(a_off[i]), int(Ks[i]),
                        dpb.at(b_off[i]), int(Ns[i]), dC.at(c_off[i]), int(Ns[i])) for i in range(count)]
    plan = ug.GroupedPlan(probs, capture=True)
    ms = time_plan(plan, stream)
    plan.destroy()
    for d in (dpa, dpb, dC):
        d.free()
    tf = flop / (ms * 1e-3) / 1e12
    return {"operands": "slices of a 16 MiB A pool and a 64 MiB B pool (cache-resident)",
            "grouped_graph_ms": round(ms, 4), "grouped_tflops": round(tf, 3),
            "frac_of_single_large_gemm_rate": round(tf / fp32_single_tf, 4) if fp32_single_tf else None}


def config4_conv(stream, gemm_grouped_tf, m32_grouped_tf=None):
    """Config 4 as convolutions: the same 512 draws (M = Cout, H = W, K = 9*Cin)
    as 3x3, pad 1, stride 1 convolutions with bias + LeakyReLU, im2col
    gathered inside the grouped kernel (no column matrix is stored).  The
    GEMM shapes equal config 4's, so the rate next to config 4's grouped GEMM
    rate is the cost of the implicit gather and the fused epilogue."""
    _, Ms, HW, Ks = config4_shapes()
    count = len(Ms)
    Cin = Ks // 9
    flop = float(np.sum(2.0 * Ms * HW * HW * Ks))
    gi = np.random.Generator(np.random.PCG64(0x55474D4D14))
    px, pw = uniform(gi, 16 << 20), uniform(gi, 4 << 20)
    pb = uniform(gi, 1 << 12)
    dpx, dpw, dpb = hip.DeviceArray.from_host(px), hip.DeviceArray.from_host(pw), hip.DeviceArray.from_host(pb)
    o_off = np.concatenate([[0], np.cumsum(((Ms * HW * HW + 3) // 4) * 4)])
    dO = hip.DeviceArray(int(o_off[-1]), np.float32)
    x_off = 4 * gi.integers(0, ((16 << 20) - Cin * HW * HW) // 4)
    w_off = 4 * gi.integers(0, ((4 << 20) - Ms * Ks) // 4)
    b_off = gi.integers(0, (1 << 12) - Ms)
    convs = [ug.ConvProblem(dpx.at(x_off[i]), int(Cin[i]), int(HW[i]), int(HW[i]), dpw.at(w_off[i]), 3, 1, 1,
                            dO.at(o_off[i]), int(Ms[i]), dpb.at(b_off[i]), ug.ACT_LEAKY_RELU, 0.1)
             for i in range(count)]
    e0, e1 = hip.Event(), hip.Event()

    def run_mode(mode):
        plan = ug.GroupedPlan(convs, mode=mode, capture=True)
        tuned = plan.tune()
        warm(lambda: plan.run(stream), stream)
        reps = 10
        e0.record(stream)
        for _ in range(reps):
            plan.run(stream)
        e1.record(stream)
        e1.synchronize()
        ms = e0.elapsed_ms(e1) / reps
        plan.destroy()
        return ug.grouped_variants(mode)[tuned], ms, check()

    def check():
        return check_convs(dO.download(), px, pw, pb, Cin, HW, Ms, x_off, w_off, b_off, o_off)

    tuned_name, ms, worst = run_mode(ug.MODE_FP32)
    m32_name, ms_m32, worst_m32 = run_mode(ug.MODE_FP32_MFMA)
    tf = flop / (ms * 1e-3) / 1e12
    tf_m32 = flop / (ms_m32 * 1e-3) / 1e12
    r = {"problems": count, "gflop": round(flop / 1e9, 2), "tuned_variant": tuned_name,
         "grouped_graph_ms": round(ms, 4), "grouped_tflops": round(tf, 3),
         "vs_grouped_gemm_same_shapes": round(tf / gemm_grouped_tf, 4) if gemm_grouped_tf else None,
         "checked_problems_worst_err_over_bound": worst,
         "fp32_mfma": {"tuned_variant": m32_name, "grouped_graph_ms": round(ms_m32, 4),
                       "grouped_tflops": round(tf_m32, 3),
                       "vs_grouped_gemm_same_shapes": round(tf_m32 / m32_grouped_tf, 4) if m32_grouped_tf else None,
                       "checked_problems_worst_err_over_bound": worst_m32},
         "note": "3x3 pad-1 convolutions + bias + LeakyReLU(0.1), implicit im2col; GEMM shapes of config 4"}
    log(f"[config4-conv] grouped implicit conv {tf:.1f} TFLOP/s ({ms:.3f} ms); on FP32 MFMA {tf_m32:.1f} TFLOP/s")
    for d in (dpx, dpw, dpb, dO):
        d.free()
    e0.destroy()
    e1.destroy()
    return r


def check_convs(out, px, pw, pb, Cin, HW, Ms, x_off, w_off, b_off, o_off):
    """Worst error over the plain FP32 bound of the four smallest convolutions
    against a direct FP64 convolution (numpy)."""
    worst = 0.0
    for i in np.argsort(Ms * HW * HW * Cin)[:4]:
        c, hw, m = int(Cin[i]), int(HW[i]), int(Ms[i])
        x = px[x_off[i]:x_off[i] + c * hw * hw].reshape(c, hw, hw).astype(np.float64)
        wk = pw[w_off[i]:w_off[i] + m * c * 9].reshape(m, c, 3, 3).astype(np.float64)
        b = pb[b_off[i]:b_off[i] + m].astype(np.float64)
        xp = np.zeros((c, hw + 2, hw + 2))
        xp[:, 1:-1, 1:-1] = x
        ref = np.zeros((m, hw, hw))
        sc = np.zeros((m, hw, hw))
        for a in range(3):
            for bb in range(3):
                win = xp[:, a:a + hw, bb:bb + hw]
                ref += np.einsum("oc,cyx->oyx", wk[:, :, a, bb], win)
                sc += np.einsum("oc,cyx->oyx", np.abs(wk[:, :, a, bb]), np.abs(win))
        ref = ref.reshape(m, -1) + b[:, None]
        ref = np.where(ref > 0, ref, 0.1 * ref)
        sc = sc.reshape(m, -1) + np.abs(b)[:, None]
        got = out[o_off[i]:o_off[i] + m * hw * hw].reshape(m, -1)
        worst = max(worst, float(np.max(np.abs(got - ref) / (2 * (c * 9 + 1) * 2.0 ** -24 * sc))))
    return worst


def blas12(stream):
    """BLAS-1/2 helpers (ugemm.h:76-160) against the HBM roofline: axpy moves
    3 words per element (read x, read y, write y); gemv reads A once, x once
    and y once and writes y."""
    g = np.random.Generator(np.random.PCG64(0x55474D4D07))
    res = {}

    def run(fn, reps=10):
        warm(fn, stream)
        e0, e1 = hip.Event(), hip.Event()
        e0.record(stream)
        for _ in range(reps):
            fn()
        e1.record(stream)
        e1.synchronize()
        ms = e0.elapsed_ms(e1) / reps
        e0.destroy()
        e1.destroy()
        return ms

    for name, dt, n in (("saxpy", np.float32, 1 << 28), ("daxpy", np.float64, 1 << 27)):
        x = hip.DeviceArray.from_host(g.standard_normal(n).astype(dt))
        y = hip.DeviceArray.from_host(g.standard_normal(n).astype(dt))
        ms = run(lambda: ug.axpy_dev(n, 0.5, x, 1, y, 1, double=dt == np.float64, stream=stream))
        gbs = 3.0 * n * np.dtype(dt).itemsize / (ms * 1e-3) / 1e9
        res[f"{name}_{n}"] = {"ms": round(ms, 4), "GB_per_s": round(gbs, 1), "frac_of_hbm_peak": round(gbs / HBM_GBPS, 4)}
        log(f"[blas12] {name} N={n}: {gbs:.0f} GB/s")
        x.free()
        y.free()
    for name, dt, M, N in (("sgemv", np.float32, 16384, 16384), ("dgemv", np.float64, 16384, 8192)):
        A = hip.DeviceArray.from_host(g.standard_normal(M * N).astype(dt))
        for trans in "NT":
            rows, cols = (M, N) if trans == "N" else (N, M)
            x = hip.DeviceArray.from_host(g.standard_normal(N).astype(dt))
            y = hip.DeviceArray.from_host(g.standard_normal(M).astype(dt))
            ms = run(lambda: ug.gemv_dev(trans, M, N, 1.0, A, rows, x, 1, 0.5, y, 1, double=dt == np.float64,
                                         stream=stream))
            nbytes = (M * N + N + 2 * M) * np.dtype(dt).itemsize
            gbs = nbytes / (ms * 1e-3) / 1e9
            res[f"{name}_{trans}_{M}x{N}"] = {"ms": round(ms, 4), "GB_per_s": round(gbs, 1),
                                              "frac_of_hbm_peak": round(gbs / HBM_GBPS, 4)}
            log(f"[blas12] {name} {trans} {M}x{N}: {gbs:.0f} GB/s")
            x.free()
            y.free()
        A.free()
    return res


def split_k(stream):
    """Few tiles, long K: automatic split-K against one split (FP32, BF16x3,
    FP64), with the split result's error bound checked on a row sample."""
    g = np.random.Generator(np.random.PCG64(0x55474D4D06))
    res = {}
    for (M, N, K) in ((256, 256, 65536), (1024, 1024, 16384)):
        A, B = g.standard_normal((M, K), dtype=np.float32), g.standard_normal((K, N), dtype=np.float32)
        rows = np.arange(0, M, max(1, M // 16))
        exact = A[rows].astype(np.float64) @ B.astype(np.float64)
        scale = np.abs(A[rows].astype(np.float64)) @ np.abs(B.astype(np.float64))
        key = f"{M}x{N}x{K}"
        res[key] = {}
        for form in ("fp32", "bf16x3", "fp64"):
            if form == "fp64":
                dA, dB = hip.DeviceArray.from_host(A.astype(np.float64)), hip.DeviceArray.from_host(B.astype(np.float64))
                dC, mid = hip.DeviceArray((M, N), np.float64), ug.MODE_DGEMM

                def call():
                    ug.dgemm_dev("R", "N", "N", M, N, K, 1.0, dA, K, dB, N, 0.0, dC, N, stream=stream)
            else:
                dA, dB = hip.DeviceArray.from_host(A), hip.DeviceArray.from_host(B)
                dC, mid = hip.DeviceArray((M, N), np.float32), ug.MODES[form]

                def call():
                    ug.sgemm_dev("R", "N", "N", M, N, K, 1.0, dA, K, dB, N, 0.0, dC, N, mode=mid, stream=stream)
            r = {}
            for label, sp in (("one_split", 1), ("auto", 0)):
                ug.force_splits(mid, sp)
                try:
                    ms, _, _ = timed(call, 10, 2, stream, 250.0)
                finally:
                    ug.force_splits(mid, 0)
                r[label + "_tflops"] = round(2.0 * M * N * K / (ms * 1e-3) / 1e12, 3)
            got = dC.download()[rows].astype(np.float64)
            r["auto_max_err_over_scale"] = float(np.max(np.abs(got - exact) / np.maximum(scale, 1e-300)))
            res[key][form] = r
            log(f"[split_k] {key} {form}: one split {r['one_split_tflops']:.1f}, auto {r['auto_tflops']:.1f} TFLOP/s")
            for d in (dA, dB, dC):
                d.free()
    return res


def host_path():
    """Host-pointer calls, copies included (the sgemm_ocl-style use of
    sgemm_ocl2.h:166-219): sgemm_test.c's own workload (M=1023, N=1000,
    K=1023, alpha=1, beta=0, RNN/RNT/RTN, 20 calls each, sgemm_test.c:168-172),
    timed by the host clock as that harness does, and one 8192^3 call of the
    uut entry sgemm_hip.  FLOP/s counts 2MNK per call."""
    L = ug.load()
    g = np.random.Generator(np.random.PCG64(0x55474D4D08))
    M, N, K, times = 1023, 1000, 1023, 20
    A = uniform(g, (M * K,))
    B = uniform(g, (K * N,))
    C = np.zeros(M * N, np.float32)
    res = {}
    for ta, tb, name in (("N", "N", "rnn"), ("N", "T", "rnt"), ("T", "N", "rtn")):
        L.sgemm_hip_packed(ta.encode(), tb.encode(), M, N, K, 1.0, A.ctypes.data, B.ctypes.data, 0.0, C.ctypes.data)
        t0 = time.perf_counter()
        for _ in range(times):
            L.sgemm_hip_packed(ta.encode(), tb.encode(), M, N, K, 1.0, A.ctypes.data, B.ctypes.data, 0.0,
                               C.ctypes.data)
        dt = (time.perf_counter() - t0) / times
        if L.ugemm_hip_last_error() != 0:
            res[name] = {"error": L.ugemm_hip_last_error_message().decode()}
            continue
        res[f"sgemm_test_{name}_{M}x{N}x{K}"] = {"ms_per_call": round(dt * 1e3, 4),
                                                  "GFLOP_per_s": round(2.0 * M * N * K / dt / 1e9, 1)}
    n = 8192
    A = uniform(g, (n, n))
    B = uniform(g, (n, n))
    C = np.zeros((n, n), np.float32)
    L.sgemm_hip(b"R", b"N", b"N", 1024, 1024, 1024, 1.0, A.ctypes.data, n, B.ctypes.data, n, 0.0, C.ctypes.data, n)
    t0 = time.perf_counter()
    L.sgemm_hip(b"R", b"N", b"N", n, n, n, 1.0, A.ctypes.data, n, B.ctypes.data, n, 0.0, C.ctypes.data, n)
    dt = time.perf_counter() - t0
    res[f"sgemm_hip_uut_{n}^3"] = {"ms_per_call": round(dt * 1e3, 3), "TFLOP_per_s": round(2.0 * n ** 3 / dt / 1e12, 2),
                                   "host_GB_moved": round(3 * n * n * 4 / 1e9, 3)}
    log(f"[host] {json.dumps(res)}")
    return res


def config1_cpu():
    """Config 1: the reference's CPU paths at 1024^3 (row-major NN, alpha 1,
    beta 0, U[-1,1) from seed 0x55474D4D01, C zero), one thread each, checked
    elementwise against an FP64 product: sgemm_avx (sgemm_avx256.h:392) and
    sgemm_c (gemm_cpu.h:284), compiled from the reference sources."""
    try:
        from oracle import oracle as orc
    except Exception as e:  # noqa: BLE001
        return {"error": f"oracle unavailable: {e}"}
    L = orc.ref_lib()
    if L is None:
        return {"error": "reference library not built"}
    n = 1024
    g = np.random.Generator(np.random.PCG64(0x55474D4D01))
    A, B = uniform(g, (n, n)), uniform(g, (n, n))
    exact = A.astype(np.float64) @ B.astype(np.float64)
    scale = np.abs(A.astype(np.float64)) @ np.abs(B.astype(np.float64))
    res = {}
    for name, cite in (("sgemm_avx", "sgemm_avx256.h:392"), ("sgemm_c", "gemm_cpu.h:284")):
        fn = getattr(L, name)
        C = np.zeros((n, n), np.float32)
        best = None
        for _ in range(3):
            t0 = time.perf_counter()
            fn(b"R", b"N", b"N", n, n, n, 1.0, A.ctypes.data, n, B.ctypes.data, n, 0.0, C.ctypes.data, n)
            dt = time.perf_counter() - t0
            best = dt if best is None else min(best, dt)
        r = {"source": cite, "threads": 1, "best_s": round(best, 4), "gflops": round(2.0 * n ** 3 / best / 1e9, 2),
             "max_err_over_bound": round(float(np.max(np.abs(C - exact) / (2 * (n + 1) * 2.0 ** -24 * scale))), 4)}
        r.update(err_stats(C, exact, scale))
        res[name] = r
        log(f"[config1] {name} 1024^3: {r['gflops']:.1f} GFLOP/s, worst/bound {r['max_err_over_bound']}")
    return res


def cpu_baseline(n, seconds_target, with_config1=False):
    """The reference's sgemm_avx (sgemm_avx256.h:392-455, the AVX path named
    by the workload) on a row band of the n^3 workload, one thread."""
    try:
        from oracle import oracle as orc
    except Exception as e:  # noqa: BLE001
        return {"error": f"oracle unavailable: {e}"}
    L = orc.ref_lib()
    if L is not None:
        fn, kind, fname = L.sgemm_avx, "reference", "sgemm_avx (sgemm_avx256.h:392)"
    else:
        fn, kind, fname = orc.lib().oracle_sgemm_packed, "port", "oracle_sgemm_packed (gemm_cpu.h blocking)"
    band = 256
    g = np.random.Generator(np.random.PCG64(7))
    A, B, C = uniform(g, (band, n)), uniform(g, (n, n)), uniform(g, (band, n))
    calls, t_total = 0, 0.0
    while t_total < seconds_target and calls < 64:
        t0 = time.perf_counter()
        fn(b"R", b"N", b"N", band, n, n, 1.5, A.ctypes.data, n, B.ctypes.data, n, 0.5, C.ctypes.data, n)
        t_total += time.perf_counter() - t0
        calls += 1
    tflops = 2.0 * band * n * n * calls / t_total / 1e12
    cpu = platform.machine()
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                cpu = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    res = {"value": round(tflops, 6), "unit": "TFLOP/s", "cores": 1, "kind": kind,
           "sample": f"{fname}, R/N/N, alpha=1.5 beta=0.5, a {band}-row band of C (M={band}, N=K={n}) of the "
                     f"{n}^3 workload, {calls} calls in {t_total:.1f} s, 1 thread of {cpu} (nproc={os.cpu_count()})"}
    if L is not None:
        res["all_cores"] = cpu_all_cores(L, n, A, B, seconds_target / 2, cpu)
        res["dgemm"] = cpu_dgemm(L, 4096, seconds_target / 2, cpu)
        if with_config1:
            res["config1_1024"] = config1_cpu()
    return res


def cpu_all_cores(L, n, A, B, seconds_target, cpu):
    """Every host core at once on the n^3 workload: each thread runs the
    reference's sgemm_avx on its own 256-row band of C (sgemm_avx keeps its
    scratch on the stack, sgemm_avx256.h:334, so disjoint bands are safe;
    ctypes drops the GIL during the call).  The threading is this build's
    arrangement, not the reference's (its harness is single-threaded)."""
    import concurrent.futures as cf
    threads = max(1, min(16, os.cpu_count() or 1))
    band = A.shape[0]
    g = np.random.Generator(np.random.PCG64(8))
    Cs = [uniform(g, (band, n)) for _ in range(threads)]

    def one(i):
        L.sgemm_avx(b"R", b"N", b"N", band, n, n, 1.5, A.ctypes.data, n, B.ctypes.data, n, 0.5, Cs[i].ctypes.data, n)

    rounds, t_total = 0, 0.0
    with cf.ThreadPoolExecutor(threads) as ex:
        while t_total < seconds_target and rounds < 16:
            t0 = time.perf_counter()
            list(ex.map(one, range(threads)))
            t_total += time.perf_counter() - t0
            rounds += 1
    tflops = 2.0 * band * n * n * threads * rounds / t_total / 1e12
    return {"value": round(tflops, 6), "unit": "TFLOP/s", "cores": threads, "kind": "reference",
            "sample": f"sgemm_avx (sgemm_avx256.h:392) on {threads} threads, each a {band}-row band of C of the "
                      f"{n}^3 workload, {rounds} rounds in {t_total:.1f} s, {cpu} (nproc={os.cpu_count()}); "
                      "threading is this build's arrangement"}


def cpu_dgemm(L, n, seconds_target, cpu):
    """The reference's dgemm_avx (dgemm_avx.h:844-923) on a row band of the
    n^3 FP64 workload (R/N/N, alpha = 1, beta = 0, normal(0,1) inputs), one
    thread: dgemm_avx packs into static buffers, so it is not threaded."""
    band = 128
    g = np.random.Generator(np.random.PCG64(9))
    A, B = g.standard_normal((band, n)), g.standard_normal((n, n))
    C = np.zeros((band, n))
    calls, t_total = 0, 0.0
    while t_total < seconds_target and calls < 64:
        t0 = time.perf_counter()
        L.dgemm_avx(b"R", b"N", b"N", band, n, n, 1.0, A.ctypes.data, n, B.ctypes.data, n, 0.0, C.ctypes.data, n)
        t_total += time.perf_counter() - t0
        calls += 1
    tflops = 2.0 * band * n * n * calls / t_total / 1e12
    return {"value": round(tflops, 6), "unit": "TFLOP/s", "cores": 1, "kind": "reference",
            "sample": f"dgemm_avx (dgemm_avx.h:844), R/N/N, a {band}-row band of C (M={band}, N=K={n}) of the "
                      f"{n}^3 FP64 workload, {calls} calls in {t_total:.1f} s, 1 thread of {cpu}"}


def load_traffic(form):
    """HBM bytes per launch of the headline core kernel from the committed
    rocprofv3 --pmc summary (FETCH_SIZE + WRITE_SIZE, calibrated), if present."""
    p = os.path.join(ROOT, "profiles", "traffic.json")
    try:
        return json.load(open(p)).get(form)
    except (OSError, ValueError):
        return None


def load_counters(form):
    """Counter figures of the form's core kernel from the committed rocprofv3
    --pmc summary (counted FLOPs, shader clock under load, MFMA busy), if present."""
    p = os.path.join(ROOT, "profiles", "flop_counters.json")
    try:
        return json.load(open(p)).get(form)
    except (OSError, ValueError):
        return None


# Left out of the printed line (whole, 28 KB: readers that keep the last 12 KB
# of an output lost its start).  Every figure stands in the [detail] line on stderr.
SECTIONS = ("config2_grid", "config3", "config4_batched", "config4_as_convolutions", "split_k", "blas12",
            "host_pointer_path", "config5_precision_ladder")
DETAIL = {"ms_median", "ms_min", "wall_s", "max_abs_err", "max_err_over_bound_scale", "core_kernel", "core_ms",
          "frac_of_fp32_vector_peak"}
SECTION_DETAIL = DETAIL | {"max_rel_err", "rms_abs_err", "core_tflops", "roofline_peak", "mfma_issue_frac", "note",
                           "mfma_utilisation", "ms_per_call", "operands", "resident_operand_bytes", "gemms_per_s",
                           "frac_of_single_large_gemm_rate"}


def summary(line):
    """The line with sections and forms cut to their main figures, numbers to five digits."""
    def cut(x, drop):
        if isinstance(x, dict):
            return {k: cut(v, drop) for k, v in x.items() if k not in drop}
        if isinstance(x, list):
            return [cut(v, drop) for v in x]
        return float(f"{x:.5g}") if isinstance(x, float) else x
    out = dict(line, forms=cut(line["forms"], DETAIL))
    out.update({k: cut(line[k], SECTION_DETAIL) for k in SECTIONS if k in line})
    if "config2_grid" in out:   # 27 cells: rate and mean relative error of each
        out["config2_grid"] = {k: [c["tflops"], c["mean_rel_err"]] if "mean_rel_err" in c else c
                               for k, c in out["config2_grid"].items()}
    return out


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    # 50 untimed headline calls (~0.13 s of BF16x3 at 8192^3): the clock
    # reaches its sustained level before the timed steps start.
    ap.add_argument("--warmup", type=int, default=50)
    ap.add_argument("--size", type=int, default=8192)
    ap.add_argument("--forms", default="fp16x3,fp32,bf16x3,fp32_mfma,bf16x6,bf16x1,fp8")
    # The form timed with exactly --warmup untimed calls and reported as
    # `value` when it meets the metric's error clause; otherwise the fastest
    # form that does (plain FP32 when none does).
    ap.add_argument("--headline", default="fp16x3")
    ap.add_argument("--no-grid", action="store_true", help="skip config 2's 2048/4096/8192 x NN/NT/TN grid")
    ap.add_argument("--only", default="", help="comma list of the sections to run after the headline forms "
                    "(grid, config3, config4, conv, splitk, blas12, host, config5); default: all")
    ap.add_argument("--quick", action="store_true", help="headline forms only")
    ap.add_argument("--dgemm", action="store_true", help="with --quick: also the 4096^3 DGEMM")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--cpu-seconds", type=float, default=10.0)
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="also run a 1 GiB device-to-device copy (HBM counter calibration under rocprofv3 --pmc)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU: this backend is a single-GPU GEMM library (multi-GPU sharding is "
              f"design-only); --gpus {args.gpus} is not supported", file=sys.stderr)
        sys.exit(2)
    if int(os.environ.get("WORLD_SIZE", "1")) > 1:
        print("bench.py runs as one process on one GPU", file=sys.stderr)
        sys.exit(2)

    n = args.size
    alpha, beta = 1.5, 0.5
    ug.init(0, 0)
    stream = hip.Stream()
    g = np.random.Generator(np.random.PCG64(0x55474D4D02))
    A, B, C0 = uniform(g, (n, n)), uniform(g, (n, n)), uniform(g, (n, n))
    rows = np.sort(np.random.Generator(np.random.PCG64(3)).choice(n, 64, replace=False))
    forms = [f for f in args.forms.split(",") if f]
    res = sgemm_forms(n, A, B, C0, alpha, beta, forms, args.steps, args.warmup, stream, rows, "config2",
                      headline=args.headline)
    del A, B, C0

    timed_forms = [k for k, v in res.items() if "tflops" in v]
    if not timed_forms:
        print("bench.py: no form ran", file=sys.stderr)
        sys.exit(1)
    # The metric's error clause: max and mean relative error vs FP64 no worse
    # than the plain FP32 kernel's on the same inputs.
    target = {}
    if "fp32" in res and "tflops" in res["fp32"]:
        p = res["fp32"]
        target = {k: {"speedup": round(v["tflops"] / p["tflops"], 3),
                      "max_rel_err_ratio": round(v["max_rel_err"] / p["max_rel_err"], 3),
                      "mean_rel_err_ratio": round(v["mean_rel_err"] / p["mean_rel_err"], 3),
                      "error_no_worse_than_fp32": bool(v["max_rel_err"] <= p["max_rel_err"]
                                                       and v["mean_rel_err"] <= p["mean_rel_err"]),
                      "met": bool(v["tflops"] >= 3 * p["tflops"] and v["max_rel_err"] <= p["max_rel_err"]
                                  and v["mean_rel_err"] <= p["mean_rel_err"])}
                  for k, v in res.items() if k != "fp32" and "tflops" in v and "max_rel_err" in v}
    accurate = [k for k, v in target.items() if v["error_no_worse_than_fp32"]]
    if args.headline in accurate or (args.headline == "fp32" and "fp32" in timed_forms):
        head = args.headline
    elif accurate:
        head = max(accurate, key=lambda k: res[k]["tflops"])
    else:
        head = "fp32" if "fp32" in timed_forms else timed_forms[0]
    h = res[head]
    peak_key, mult = FORM_PEAK[head]
    flop = 2.0 * n ** 3
    core_tf = h["core_tflops"] or h["tflops"]
    roof = {"bound": "mfma", "kernel": h["core_kernel"], "achieved": core_tf,
            "peak": PEAK[peak_key], "unit": "TFLOP/s", "frac": round(core_tf / PEAK[peak_key], 4),
            "traffic": load_traffic(head),
            "achieved_is": "algorithmic 2*M*N*K flop per launch / average core-kernel duration (HIP events)",
            "mfma_issue_frac": round(core_tf * mult / PEAK[peak_key], 4),
            "frac_of_fp32_vector_peak": round(core_tf / PEAK["fp32_vector"], 4)}
    sustained = mfma_sustained()
    elem = {"fp16x3": "f16", "bf16x3": "bf16", "bf16x6": "bf16", "bf16x1": "bf16"}.get(head)
    if elem:
        # What the core reaches of the matrix-core rate this device sustains
        # under its power limit (all three products of the split counted).
        roof["sustained_mfma_peak"] = sustained[elem]
        roof["mfma_issue_frac_of_sustained"] = round(core_tf * mult / sustained[elem], 4)
    cnt = load_counters(head)
    if cnt:
        # From profiles/gemm_flop_counters.md: the clock the kernel runs at under
        # load and the fraction of cycles its MFMA pipes are busy.
        roof["counters"] = {"counted_flops_per_launch": cnt["flops"], "clock_ghz_under_load": cnt["clock_ghz"],
                            "mfma_busy": cnt["mfma_busy"],
                            "mfma_issue_frac_at_that_clock": round(core_tf * mult / (PEAK[peak_key] *
                                                                                     cnt["clock_ghz"] / 2.4), 4)}

    line = {
        "metric": "SGEMM TFLOP/s at 8192^3: plain FP32 vs BF16x3-MFMA at FP32-level error",
        "value": h["tflops"], "unit": "TFLOP/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": h["ms_per_call"], "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": DTYPE[head],
        "data": "synthetic: U[-1,1) 24-bit from PCG64 seed 0x55474D4D02, resident in HBM",
        "config": {"workload": f"sgemm {n}x{n}x{n} row-major NN alpha={alpha} beta={beta}; step = one GEMM call "
                               f"(operand preparation + core) in form {head}",
                   "M": n, "N": n, "K": n, "layout": "NN", "form": head,
                   "form_rule": "the --headline form (fp16x3) if its max and mean relative error vs FP64 are no "
                                "worse than plain FP32's on the same inputs, else the fastest form that meets "
                                "that; BF16x3 (a 2-way bf16 split keeps 16-17 significant bits) is reported "
                                "in forms with its error ratios"},
        "forms": res,
        "roofline": roof,
        "mfma_sustained_tflops": dict(sustained, note="16x16x32 MFMAs only, on every SIMD, operands = split "
                                      "planes of U[-1,1) data; published dense peak 2516.6"),
    }
    if target:
        line["speedup_vs_plain_fp32"] = {k: round(v["tflops"] / res["fp32"]["tflops"], 3)
                                         for k, v in res.items() if "tflops" in v}
        line["error_vs_plain_fp32"] = {k: round(v["rms_abs_err"] / res["fp32"]["rms_abs_err"], 3)
                                       for k, v in res.items() if "rms_abs_err" in v}
        # The throughput/accuracy target: >= 3x plain FP32 TFLOP/s with max and
        # mean relative error vs FP64 no worse than plain FP32's.
        line["target_3x_at_fp32_error"] = target
        # The same ratio against the FP32-MFMA form, the fastest FP32-class
        # kernel here (not the plain vector-FMA kernel the target names).
        if "fp32_mfma" in res:
            line["speedup_vs_fp32_mfma"] = {k: round(v["tflops"] / res["fp32_mfma"]["tflops"], 3)
                                            for k, v in res.items() if "tflops" in v}
    if args.calibrate_copy:
        nbytes = 1 << 30
        src, dst = hip.DeviceArray(nbytes // 4, np.float32), hip.DeviceArray(nbytes // 4, np.float32)
        hip.check(hip.lib().hipMemcpy(dst.ptr, src.ptr, nbytes, hip.D2D), "calibration copy")
        hip.synchronize()
        line["calibration_copy_bytes"] = nbytes
        src.free()
        dst.free()
    if args.quick and args.dgemm:
        line["dgemm_4096"] = dgemm_4096(stream, args.steps)
    only = set(x for x in args.only.split(",") if x)
    want = (lambda sec: not args.quick and (not only or sec in only))
    if want("grid") and not args.no_grid:
        line["config2_grid"] = config2_grid(stream, args.steps)
    if want("config3"):
        line["config3"] = config3(stream, args.steps, args.warmup)
    if want("config4"):
        fp32_tf = res.get("fp32", {}).get("tflops")
        line["config4_batched"] = config4(stream, fp32_tf, {k: v.get("tflops") for k, v in res.items()})
    if want("conv"):
        c4 = line.get("config4_batched", {})
        line["config4_as_convolutions"] = config4_conv(stream, c4.get("grouped_tflops"),
                                                       c4.get("fp32_mfma_grouped", {}).get("grouped_tflops"))
    if want("splitk"):
        line["split_k"] = split_k(stream)
    if want("blas12"):
        line["blas12"] = blas12(stream)
    if want("host"):
        line["host_pointer_path"] = host_path()
    if want("config5"):
        g5 = np.random.Generator(np.random.PCG64(0x55474D4D05))
        A5, B5 = wide(g5, (n, n)), wide(g5, (n, n))
        C5 = np.zeros((n, n), np.float32)
        line["config5_precision_ladder"] = sgemm_forms(n, A5, B5, C5, 1.0, 0.0, ["fp32", "bf16x3", "fp16x3",
                                                                                  "fp32_mfma", "bf16x6", "bf16x1",
                                                                                  "fp8"],
                                                       max(5, args.steps // 4), 2, stream, rows, "config5")
        del A5, B5, C5
    if not args.no_cpu:
        line["cpu_baseline"] = cpu_baseline(n, args.cpu_seconds, with_config1=not args.quick)
    log("[detail] " + json.dumps(line))
    print(json.dumps(summary(line)), flush=True)


if __name__ == "__main__":
    main()
