#!/usr/bin/env python3
"""Benchmark of the interleaved block-cyclic FFT + stencil path on one MI355X.

Workload (default): 2D N=8192, P=4 (16 virtual ranks), B=32.  One step is the
round trip of the reference's example() (zmodel/main.cu:50-80): 5-point
Laplacian (h = 1/N) -> forward 2D FFT -> inverse 2D FFT scaled 1/N^2, on a
seeded smooth field (256 random Fourier modes with |k| <= N/8, amplitudes
N(0,1)/(1+|k|^2), uniform phases, plus 1e-3 uniform noise) held in HBM.  The
step runs as zm_laplace_forward (the Laplacian formed inside the forward
transform's x pass: 3 kernel sweeps instead of 4, bit for bit the same
result) then zm_inverse; --separate times the reference's three calls
instead, and the other chain is always timed beside the headline
(`other_chain`).

Prints one JSON line on stdout (diagnostics go to stderr):
  value        FFT GFLOP/s, 5 N^2 log2(N^2) per transform, two transforms per
               step, FP32 vector-ALU path
  roofline     the step's dominant kernel (the fused direction pass): its
               launch durations come from HIP events recorded after each
               launch on its stream, in a second timed pass of the same steps
  errors       relative L2 / max error of every FP32 output against the FP64
               GPU path on the same FP32-rounded input
  fp32_mfma    the same step with the radix-16 stages as split-precision MFMA
               GEMMs: step time, line-pass time, errors
  derivatives  dx4 / dy4 (dz4 in 3D) launch times and bandwidth
  config_3d    the 3D configuration (512^3, P=2, B=16): FP32 and FP64 steps
  library_fft  the FFT round trip alone beside torch.fft.fftn + ifftn (rocFFT)
               on the natural layout of the same field and precision
  cpu_baseline the stand-in for the reference CPU path (heFFTe + FFTW is not in
               the image): scipy.fft (pocketfft) + a numpy Laplacian on the host
               cores, on the same field; the FP64 GPU path is checked against
               its output, and the FP64 C oracle (a port) is timed beside it
"""
from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def rel_errors(a, ref, torch):
    d = (a.to(torch.complex128) - ref)
    l2 = float(torch.linalg.vector_norm(d) / torch.linalg.vector_norm(ref))
    mx = float(d.abs().max() / ref.abs().max())
    return {"rel_l2": l2, "rel_max": mx}


def run_steps(plan, x, lap, y, z, scratch, n, steps, torch, stream, fused=True):
    """One step = the Laplacian (h = 1/N), the forward transform and the
    inverse transform (1/N^d).  fused: zm_laplace_forward then zm_inverse
    (on FP32 plans with the fused pass the Laplacian is formed inside the
    forward transform's x pass); otherwise the three calls of the reference's
    example() (zm_laplace, zm_forward, zm_inverse), with the Laplacian
    written to `lap`."""
    dims = plan.shape.dims
    for _ in range(steps):
        if fused:
            plan.laplace_forward(x, float(n * n), out=y, scratch=scratch, stream=stream)
        else:
            plan.laplace(x, scale=float(n * n), out=lap, stream=stream)
            plan.forward(lap, out=y, scratch=scratch, stream=stream)
        plan.inverse(y, 1.0 / float(n) ** dims, out=z, scratch=scratch, stream=stream)


def time_path(plan, x, n, steps, warmup, torch, label, fused=True):
    """Time exactly `steps` steps with no per-launch instrumentation (the step
    time and `value`), then the same `steps` again with the plan's per-launch
    HIP events, one recorded on the launch stream after every kernel (the
    stage breakdown and the dominant kernel's launch durations).  Returns the
    step's outputs (Laplacian, forward, round trip); the fused step does not
    write its Laplacian, which is computed after the timed steps."""
    lap = torch.empty_like(x)
    y = torch.empty_like(x)
    z = torch.empty_like(x)
    scratch = torch.empty(plan.scratch_bytes // x.element_size(), dtype=x.dtype, device="cuda")
    stream = torch.cuda.current_stream()
    run_steps(plan, x, lap, y, z, scratch, n, warmup, torch, stream, fused)
    torch.cuda.synchronize()

    def timed(instrumented):
        if instrumented:
            plan.timing_reset()
            plan.timing(True)
        start = torch.cuda.Event(enable_timing=True)
        stop = torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        start.record(stream)
        run_steps(plan, x, lap, y, z, scratch, n, steps, torch, stream, fused)
        stop.record(stream)
        torch.cuda.synchronize()
        wall = time.perf_counter() - t0
        if instrumented:
            plan.timing(False)
        return start.elapsed_time(stop) / steps, wall

    ms, wall = timed(False)
    ms_instr, _ = timed(True)
    # a stage done inside another stage's launch is counted with no time of its
    # own: it is no launch and no kernel sweep
    stages = {k: (c, t) for k, (c, t) in plan.timing_read().items() if t > 0}
    plan.timing_reset()
    if fused:
        plan.laplace(x, scale=float(n * n), out=lap, stream=stream)
        torch.cuda.synchronize()
    log(f"{label}{' (fused Laplacian)' if fused else ''}: {ms:.3f} ms/step (wall {1e3 * wall / steps:.3f} ms/step; "
        f"with per-launch events {ms_instr:.3f}); stages "
        + ", ".join(f"{k}: {c} x {t / c:.3f} ms" for k, (c, t) in stages.items()))
    time_path.last_instrumented = ms_instr
    return ms, stages, (lap, y, z)


def time_graph(plan, x, n, steps, torch, fused=True):
    """One step captured in a HIP graph (torch.cuda.graph on the plan's
    stream-ordered launches), replayed `steps` times."""
    lap, y, z = torch.empty_like(x), torch.empty_like(x), torch.empty_like(x)
    scratch = torch.empty(plan.scratch_bytes // x.element_size(), dtype=x.dtype, device="cuda")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        run_steps(plan, x, lap, y, z, scratch, n, 2, torch, None, fused)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        run_steps(plan, x, lap, y, z, scratch, n, 1, torch, None, fused)
    for _ in range(3):
        g.replay()
    torch.cuda.synchronize()
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    ev0.record()
    for _ in range(steps):
        g.replay()
    ev1.record()
    torch.cuda.synchronize()
    ms = ev0.elapsed_time(ev1) / steps
    log(f"graph replay: {ms:.4f} ms/step")
    return ms


def library_fft_comparison(plan, x, n, steps, warmup, torch):
    """The FFT round trip alone (forward, then inverse scaled 1/N^d) on the
    packed layout against torch.fft.fftn / ifftn (hipFFT over rocFFT) on the
    natural layout of the same field and precision: the role of the
    reference's heFFTe + cuFFT example (heffte/heffte_example_cuda.cpp).
    Forward errors of both are taken against the FP64 library transform."""
    dims = plan.shape.dims
    axes = tuple(range(dims))
    nat = plan.packed_to_natural(x).reshape((n,) * dims)
    y, z = torch.empty_like(x), torch.empty_like(x)
    scratch = torch.empty(plan.scratch_bytes // x.element_size(), dtype=x.dtype, device="cuda")
    stream = torch.cuda.current_stream()
    scale = 1.0 / float(n) ** dims

    def ours(k):
        for _ in range(k):
            plan.forward(x, out=y, scratch=scratch, stream=stream)
            plan.inverse(y, scale, out=z, scratch=scratch, stream=stream)

    def lib(k):
        for _ in range(k):
            f = torch.fft.fftn(nat, dim=axes)
            torch.fft.ifftn(f, dim=axes)

    out = {}
    for name, fn in (("ours", ours), ("library", lib)):
        fn(warmup)
        torch.cuda.synchronize()
        ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        ev0.record(stream)
        fn(steps)
        ev1.record(stream)
        torch.cuda.synchronize()
        out[name] = ev0.elapsed_time(ev1) / steps
    ref = torch.fft.fftn(nat.to(torch.complex128), dim=axes).reshape(-1)
    tab = plan.reciprocal_index_table()
    ours_nat = torch.empty_like(y)
    ours_nat[tab] = y
    del tab
    err_ours = rel_errors(ours_nat, ref, torch)
    del ours_nat
    err_lib = rel_errors(torch.fft.fftn(nat, dim=axes).reshape(-1), ref, torch)
    res = {
        "library": f"torch.fft.fftn + ifftn (hipFFT/rocFFT), natural {n}^{dims} layout, {str(x.dtype)[6:]}",
        "ms_per_round_trip": round(out["library"], 4),
        "ours_ms_per_round_trip": round(out["ours"], 4),
        "speedup_vs_library": round(out["library"] / out["ours"], 3),
        "forward_errors_vs_fp64_library": {"ours": err_ours, "library": err_lib},
    }
    log(f"library FFT comparison: {json.dumps(res)}")
    return res


def time_derivatives(plan, x, n, reps, torch):
    """Average launch time of dx4 / dy4 (and dz4 on a 3D plan) with delta = 1/N,
    from the plan's per-launch HIP events on the current stream; one read and
    one write of the field per launch."""
    stream = torch.cuda.current_stream()
    out = torch.empty_like(x)
    names = ("dx4", "dy4", "dz4") if plan.shape.dims == 3 else ("dx4", "dy4")
    res = {}
    for name in names:
        fn = getattr(plan, name)
        for _ in range(2):
            fn(x, 1.0 / n, out=out, stream=stream)
        torch.cuda.synchronize()
        plan.timing_reset()
        plan.timing(True)
        for _ in range(reps):
            fn(x, 1.0 / n, out=out, stream=stream)
        plan.timing(False)
        c, t = plan.timing_read()["deriv"]
        plan.timing_reset()
        avg = t / c
        nbytes = 2 * x.numel() * x.element_size()
        res[name] = {"avg_launch_ms": round(avg, 4), "achieved_gbs": round(nbytes / (avg * 1e-3) / 1e9, 1),
                     "frac": round(nbytes / (avg * 1e-3) / 1e9 / HBM_PEAK_GBS, 4)}
    log(f"derivatives: {json.dumps(res)}")
    return res


def stage_roofline(stages, nbytes):
    """Per-stage average launch time and bandwidth (one read + one write of
    `nbytes` per launch for every stage kernel of the fused path)."""
    out = {}
    for k, (c, t) in stages.items():
        avg = t / c
        out[k] = {"avg_launch_ms": round(avg, 4), "achieved_gbs": round(2 * nbytes / (avg * 1e-3) / 1e9, 1)}
    return out


def cpu_baseline(nat_in, dims, n, p, b, seed, gpu64, plan64, torch, with_port=True):
    """The reference CPU path's stand-in, on the same field as the GPU legs.

    The reference's CPU path is heFFTe with FFTW (heffte/heffte_example_fftw.cpp),
    which is not in the image.  Stand-in: a numpy periodic Laplacian plus
    scipy.fft fftn / ifftn (pocketfft, FP64, one worker per host core) on the
    natural layout of the same seeded field.  Median of 5 timed steps after a
    warm-up; the forward transform alone is timed as heFFTe's example does
    (heffte_example_fftw.cpp:78-87).  `nat_in` is the natural-layout input of
    the FP64 GPU path `gpu64` (Laplacian, forward, round trip), whose forward
    output and round trip are compared with the stand-in's
    (heffte_example_fftw.cpp:105-124 checks its own round trip the same way).
    Beside it, the FP64 C oracle (a port of the reference path) runs one full
    step of the same field."""
    import numpy as np
    import scipy.fft as sfft

    threads = len(os.sched_getaffinity(0))
    field = float(n) ** dims
    flops = 2 * 5.0 * field * math.log2(field)
    xn = nat_in.reshape((n,) * dims)

    def step():
        u0 = time.perf_counter()
        lap = -2.0 * dims * xn
        for ax in range(dims):
            lap += np.roll(xn, 1, ax) + np.roll(xn, -1, ax)
        lap *= float(n * n)
        u1 = time.perf_counter()
        y = sfft.fftn(lap, workers=threads)
        u2 = time.perf_counter()
        z = sfft.ifftn(y, workers=threads)
        u3 = time.perf_counter()
        return (u3 - u0, u2 - u1), (y, z)

    step()  # warm-up
    times = []
    for _ in range(5):
        t, outs = step()
        times.append(t)
        if len(times) < 5:
            del outs
    med = sorted(times)[2]
    fwd = sorted(t[1] for t in times)[2]
    y_cpu, z_cpu = outs
    # the FP64 GPU outputs in natural order
    lap64, y64, z64 = gpu64
    tab = plan64.reciprocal_index_table()
    y_nat = torch.empty_like(y64)
    y_nat[tab] = y64
    del tab
    y_gpu = y_nat.cpu().numpy().reshape((n,) * dims)
    del y_nat
    z_gpu = plan64.packed_to_natural(z64).cpu().numpy().reshape((n,) * dims)

    def errs(a, ref):
        d = a - ref
        return {"rel_l2": float(np.linalg.norm(d.ravel()) / np.linalg.norm(ref.ravel())),
                "rel_max": float(np.max(np.abs(d)) / np.max(np.abs(ref)))}

    check = {"forward": errs(y_gpu, y_cpu), "round_trip": errs(z_gpu, z_cpu)}
    del y_gpu, z_gpu, y_cpu, z_cpu, outs
    log(f"cpu stand-in ({threads} workers): step median {med[0]:.3f} s, forward {fwd:.3f} s; "
        f"FP64 GPU vs stand-in {json.dumps(check)}")
    res = {
        "value": round(flops / med[0] / 1e9, 3),
        "unit": "GFLOP/s",
        "cores": threads,
        "kind": "standin",
        "label": "stand-in for heFFTe+FFTW (the reference CPU path, not in the image): scipy.fft pocketfft FP64",
        "sample": (f"one full step (numpy periodic {2 * dims + 1}-point Laplacian, h=1/N; scipy.fft fftn; ifftn) of "
                   f"the same complex128 {n}^{dims} field on the natural layout with {threads} workers, median of 5 "
                   f"after a warm-up: {med[0]:.3f} s per step, forward alone {fwd:.3f} s"),
        "seconds_per_step": round(med[0], 4),
        "forward_seconds": round(fwd, 4),
        "fp64_gpu_vs_standin": check,
    }
    if with_port:
        import oracle
        oracle.build()
        s = oracle.Shape(dims, n, p, b)
        x = s.natural_to_real(xn)
        oracle.set_dft_mode(1)
        try:
            t0 = time.perf_counter()
            lap = s.laplace(x)
            t1 = time.perf_counter()
            y = s.forward_fft(lap)
            t2 = time.perf_counter()
            s.inverse_fft(y, scale=1.0 / field)
            t3 = time.perf_counter()
        finally:
            oracle.set_dft_mode(0)
        del lap, y, x
        log(f"cpu oracle port ({threads} threads): laplace {t1 - t0:.2f} s, forward {t2 - t1:.2f} s, "
            f"inverse {t3 - t2:.2f} s")
        res["port_oracle"] = {
            "value": round(flops / (t3 - t0) / 1e9, 3), "unit": "GFLOP/s", "cores": threads, "kind": "port",
            "sample": (f"one full step (Laplacian, forward FFT, inverse FFT) of the same field, {dims}D N={n} P={p} "
                       f"B={b}, in the FP64 C oracle (radix-2 DFT mode, OpenMP): {t3 - t0:.2f} s, forward alone "
                       f"{t2 - t1:.2f} s"),
            "seconds_per_step": round(t3 - t0, 3),
        }
    return res


def load_traffic(name):
    path = os.path.join(ROOT, "profiles", name)
    if not os.path.exists(path):
        return None
    with open(path) as f:
        return json.load(f)


KERNELS = {"line": "line_fast_kernel (fused FFT1a + exchange + twiddle + FFT1b direction pass, forward and inverse "
                   "instantiations)",
           "line_laplace": "line_fast_kernel with the 5-point Laplacian formed ahead of the forward x pass",
           "repack": "repack_tiled_kernel", "laplace": "laplace_strip_kernel",
           "stage_a": "stage_a_kernel", "stage_b": "stage_b_kernel"}


def make_field(plan64, dims, n, seed, torch):
    """The configuration's seeded field, natural layout (complex128) and packed."""
    if dims == 2:
        from stencilfft_amd.fields import mode_field_natural
        nat = mode_field_natural(n, 2, 256, n // 8, seed, noise=1e-3)
        desc = f"256 modes |k|<=N/8, amp N(0,1)/(1+|k|^2), + 1e-3 U[-1,1) noise, seed {seed}"
    else:
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        re = torch.rand(n ** 3, generator=g, device="cuda", dtype=torch.float64) * 2 - 1
        im = torch.rand(n ** 3, generator=g, device="cuda", dtype=torch.float64) * 2 - 1
        nat = torch.complex(re, im)
        del re, im
        desc = f"re, im U[-1,1) (torch CUDA generator), seed {seed}"
    return nat, plan64.natural_to_packed(nat), desc


def compare_outputs(plan, plan64, x, x64r, outs, outs64, n, torch):
    errs = {}
    for name, a, r in zip(("laplace", "forward", "round_trip"), outs, outs64):
        errs[name] = rel_errors(a, r, torch)
    derivs = ("dx4", "dy4") if plan.shape.dims == 2 else ("dx4", "dy4", "dz4")
    if plan.shape.b >= 2:
        for name in derivs:
            d32 = getattr(plan, name)(x, 1.0 / n)
            d64 = getattr(plan64, name)(x64r, 1.0 / n)
            errs[name] = rel_errors(d32, d64, torch)
            del d32, d64
    return errs


def leg_3d(args, torch, Plan):
    """The 3D configuration: 512^3, P=2, B=16, U[-1,1) field; FP32 and FP64
    steps (Laplacian 7-point, forward, inverse), stage times, errors.  The
    FP32 step is zm_laplace_forward + zm_inverse (the Laplacian formed inside
    the x pass), with the reference's three calls timed beside it; FP64 runs
    the three calls (it has no fused pass)."""
    n, p, b = 512, 2, 16
    steps = max(3, min(args.steps, 10))
    plan64 = Plan(3, n, p, b, precision="fp64")
    nat, x64, desc = make_field(plan64, 3, n, args.seed, torch)
    del nat
    plan32 = Plan(3, n, p, b, precision="fp32")
    x32 = x64.to(torch.complex64)
    del x64
    x64r = x32.to(torch.complex128)
    ms32, st32, outs32 = time_path(plan32, x32, n, steps, 2, torch, "3D fp32", True)
    ms32s, st32s, outs32s = time_path(plan32, x32, n, steps, 2, torch, "3D fp32", False)
    del outs32s
    ms64, st64, outs64 = time_path(plan64, x64r, n, steps, 2, torch, "3D fp64", False)
    errs = compare_outputs(plan32, plan64, x32, x64r, outs32, outs64, n, torch)
    del outs32, outs64
    der = time_derivatives(plan32, x32, n, 10, torch)
    field = float(n) ** 3
    flops = 2 * 5.0 * field * math.log2(field)
    res = {
        "workload": f"3D N={n} P={p} B={b} (8 virtual ranks): 7-point Laplacian -> forward FFT -> inverse FFT",
        "field": desc,
        "step_chain": (f"FP32: zm_laplace_forward, zm_inverse ({sum(c for c, _ in st32.values()) // steps} kernel "
                       f"sweeps); FP64 and fp32_three_call: zm_laplace, zm_forward, zm_inverse "
                       f"({sum(c for c, _ in st64.values()) // steps} kernel sweeps)"),
        "fp32_ms_per_step": round(ms32, 4), "fp32_gflops": round(flops / (ms32 * 1e-3) / 1e9, 1),
        "fp32_three_call_ms_per_step": round(ms32s, 4),
        "fp32_three_call_stages": stage_roofline(st32s, x32.numel() * x32.element_size()),
        "fp64_ms_per_step": round(ms64, 4), "fp64_gflops": round(flops / (ms64 * 1e-3) / 1e9, 1),
        "speedup_fp32_vs_fp64_gpu": round(ms64 / ms32, 3),
        "fp32_stages": stage_roofline(st32, x32.numel() * x32.element_size()),
        "fp64_stages": stage_roofline(st64, x64r.numel() * x64r.element_size()),
        "fp32_derivatives": der,
        "errors_fp32_vs_fp64_gpu": errs,
    }
    log(f"3D leg: {json.dumps(res)}")
    return res


def main():
    ap = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--precision", default="fp32", choices=["fp32", "fp64", "fp32_mfma"])
    ap.add_argument("--dims", type=int, default=2, choices=[2, 3])
    ap.add_argument("--n", type=int, default=None, help="default 8192 (2D) / 512 (3D)")
    ap.add_argument("--p", type=int, default=None, help="default 4 (2D) / 2 (3D)")
    ap.add_argument("--b", type=int, default=None, help="default 32 (2D) / 16 (3D)")
    ap.add_argument("--two-stage", action="store_true", help="force the two-kernel-per-direction path")
    ap.add_argument("--separate", action="store_true",
                    help="time the reference's three calls per step (Laplacian, forward, inverse) as the headline "
                         "instead of the chain with the Laplacian fused into the forward transform")
    ap.add_argument("--no-fp64", action="store_true", help="skip the FP64 comparison paths")
    ap.add_argument("--no-mfma", action="store_true", help="skip the split-precision MFMA leg")
    ap.add_argument("--no-3d", action="store_true", help="skip the 3D configuration leg")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-library-fft", action="store_true",
                    help="skip the torch.fft (rocFFT) natural-layout round-trip comparison")
    ap.add_argument("--seed", type=int, default=8192)
    ap.add_argument("--graph", action="store_true",
                    help="also time the step captured once in a HIP graph and replayed (graph_ms_per_step)")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="time a plain device-to-device copy of one N^2 complex64 field (the HBM reference "
                         "kernel the rocprof FETCH_SIZE / WRITE_SIZE counters are scaled by) and exit")
    args = ap.parse_args()

    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print(json.dumps({"error": "stencilfft-amd runs the whole P x P virtual rank grid on one GPU; "
                                   "--gpus must be 1 (multi-GPU sharding is a design note, not built)"}))
        sys.exit(2)

    import torch

    from stencilfft_amd import Plan
    if not torch.cuda.is_available():
        print(json.dumps({"error": "no GPU"}))
        sys.exit(1)

    dims = args.dims
    dflt = {2: (8192, 4, 32), 3: (512, 2, 16)}[dims]
    n = args.n or dflt[0]
    p = args.p or dflt[1]
    b = args.b or dflt[2]
    if args.copy_calibration:
        src = torch.ones(n * n, dtype=torch.complex64, device="cuda")
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        reps = 10
        ev0.record()
        for _ in range(reps):
            dst.copy_(src)
        ev1.record()
        torch.cuda.synchronize()
        ms = ev0.elapsed_time(ev1) / reps
        nbytes = 2 * src.numel() * src.element_size()
        print(json.dumps({"metric": "device-to-device copy bandwidth", "value": round(nbytes / ms / 1e6, 1),
                          "unit": "GB/s", "bytes_per_copy_read": src.numel() * src.element_size(),
                          "bytes_per_copy_write": src.numel() * src.element_size(), "ms_per_copy": round(ms, 4),
                          "frac_of_peak": round(nbytes / ms / 1e6 / HBM_PEAK_GBS, 4)}))
        return
    log(f"workload {dims}D N={n} P={p} B={b} precision={args.precision} steps={args.steps} warmup={args.warmup}")
    plan64 = Plan(dims, n, p, b, precision="fp64", two_stage=args.two_stage)
    nat64, x64, field_desc = make_field(plan64, dims, n, args.seed, torch)
    del nat64
    if args.precision == "fp64":
        plan = plan64
        x = x64
    else:
        plan = Plan(dims, n, p, b, precision=args.precision, two_stage=args.two_stage)
        x = x64.to(torch.complex64)
    del x64
    torch.cuda.synchronize()

    fused = not (args.separate or args.two_stage)
    ms, stages, outs = time_path(plan, x, n, args.steps, args.warmup, torch, args.precision, fused)
    esize = x.element_size()
    field = n ** dims
    flops = 2 * 5.0 * field * math.log2(field)
    gflops = flops / (ms * 1e-3) / 1e9
    # bytes per step: 2 sweeps per direction and FFT (pack, exchange, twiddle
    # and repack fused into adjacent loads and stores) and the textbook bound
    # (1 sweep per direction), plus one sweep for the stencil
    sweep = 2 * field * esize
    bytes_2sweep = 2 * (2 * dims) * sweep + sweep
    bytes_textbook = 2 * dims * sweep + sweep
    step_frac = bytes_2sweep / (ms * 1e-3) / 1e9 / HBM_PEAK_GBS

    # dominant kernel and its roofline: algorithmic bytes of one launch = one
    # read and one write of the field (every stage kernel here moves exactly
    # that), over its average launch duration
    dom_name, (dom_count, dom_ms) = max(stages.items(), key=lambda kv: kv[1][1])
    dom_avg = dom_ms / dom_count
    per_launch = 2 * field * esize
    achieved = per_launch / (dom_avg * 1e-3) / 1e9
    traffic = load_traffic(f"traffic_{dom_name}_n{n}_p{p}_b{b}_{args.precision}.json")
    kernel = KERNELS.get(dom_name, dom_name)
    if dom_name == "line" and plan.tiled:
        kernel = "line_pass_kernel (one whole line's FFT, pack, exchange, twiddle and repack in a pass)"
    elif dom_name == "line" and not plan.fast:
        kernel = "line_kernel (fused FFT1a + exchange + twiddle + FFT1b direction pass)"
    roofline = {
        "bound": "hbm",
        "kernel": kernel,
        "achieved": round(achieved, 1),
        "peak": HBM_PEAK_GBS,
        "unit": "GB/s",
        "frac": round(achieved / HBM_PEAK_GBS, 4),
        "traffic": traffic["bytes_per_launch"] if traffic else None,
        "bytes_per_launch": per_launch,
        "avg_launch_ms": round(dom_avg, 4),
        "launches": dom_count,
        "basis": "algorithmic bytes of one launch: one read and one write of the N^d field",
    }

    extra = {}
    if args.graph:
        extra["graph_ms_per_step"] = round(time_graph(plan, x, n, args.steps, torch, fused), 4)
    # the step's chain: zm_laplace_forward (on 2D FP32 plans with N >= 4096
    # the Laplacian is formed inside the forward transform's x pass) then
    # zm_inverse, or the reference's three calls; the other one is timed
    # beside it.  A kernel sweep is one launch that reads and writes the field.
    def sweeps_of(st):
        return sum(c for c, _ in st.values()) // args.steps
    extra["step_chain"] = {
        "fused": fused,
        "kernel_sweeps_per_step": sweeps_of(stages),
        "description": ("zm_laplace_forward then zm_inverse" if fused
                        else "zm_laplace, zm_forward, zm_inverse (zmodel/main.cu:50-78)"),
    }
    if not args.two_stage:
        ksteps = max(3, min(args.steps, 10))
        msx, stx, outsx = time_path(plan, x, n, ksteps, 2, torch, args.precision, not fused)
        del outsx
        extra["other_chain"] = {
            "fused": not fused, "ms_per_step": round(msx, 4), "gflops": round(flops / (msx * 1e-3) / 1e9, 1),
            "kernel_sweeps_per_step": sum(c for c, _ in stx.values()) // ksteps,
            "stages": stage_roofline(stx, field * esize),
        }
    if "line_laplace" in stages:
        # the fused pass does the work of two sweeps (the Laplacian's and the
        # x pass's) in one read and one write of the field; what it saves is
        # set against the two launches of the other chain
        c, t = stages["line_laplace"]
        avg = t / c
        fp = {
            "kernel": KERNELS["line_laplace"],
            "avg_launch_ms": round(avg, 4),
            "achieved_gbs": round(per_launch / (avg * 1e-3) / 1e9, 1),
            "frac": round(per_launch / (avg * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
            "basis": "one read and one write of the field per launch",
        }
        other = extra.get("other_chain", {}).get("stages", {})
        if "laplace" in other and "line" in other:
            sep = other["laplace"]["avg_launch_ms"] + other["line"]["avg_launch_ms"]
            fp["separate_laplace_plus_line_ms"] = round(sep, 4)
            fp["saved_ms_per_step"] = round(sep - avg, 4)
        extra["fused_laplace_pass"] = fp
    extra.update({
        "ms_per_step_with_launch_events": round(time_path.last_instrumented, 4),
        "stage_ms": {k: round(t / c, 4) for k, (c, t) in stages.items()},
        "stage_launches_per_step": {k: c // args.steps for k, (c, t) in stages.items()},
        "stages": stage_roofline(stages, field * esize),
        "step_bytes_2sweep": bytes_2sweep,
        "step_bytes_textbook": bytes_textbook,
        # model byte counts over the step time: with the Laplacian fused into
        # the x pass the kernels move fewer bytes than the 2-sweep model
        # counts, so that ratio can pass 1 and is not a bandwidth; the
        # bandwidth is step_hbm_frac_moved (the bytes the kernels move)
        "step_hbm_frac_2sweep": round(step_frac, 4),
        "step_hbm_frac_textbook": round(bytes_textbook / (ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
        "step_bytes_moved": extra["step_chain"]["kernel_sweeps_per_step"] * sweep,
        "step_hbm_frac_moved": round(extra["step_chain"]["kernel_sweeps_per_step"] * sweep / (ms * 1e-3) / 1e9
                                     / HBM_PEAK_GBS, 4),
    })
    moved = extra["step_hbm_frac_moved"]
    extra["target_hbm_frac"] = {"target": 0.70, "measured": moved, "met": moved >= 0.70,
                                "basis": "step_hbm_frac_moved: the bytes the step's kernels move over its time"}
    if plan.shape.b >= 2:
        extra["derivatives"] = time_derivatives(plan, x, n, 10, torch)

    outs64 = None
    if not args.no_fp64 and args.precision != "fp64":
        x64r = x.to(torch.complex128)
        # the FP64 oracle: the plain FP64 GPU path with the reference's three
        # calls (its Laplacian bit for bit the reference's); every FP32 output
        # is compared with it
        ms64s, st64s, outs64 = time_path(plan64, x64r, n, max(3, min(args.steps, 10)), 2, torch, "fp64", False)
        errs = compare_outputs(plan, plan64, x, x64r, outs, outs64, n, torch)
        errs["round_trip_vs_fp64_laplace"] = rel_errors(outs[2], outs64[0], torch)
        extra["errors_vs_fp64_gpu"] = errs
        # FP64 has no fused Laplacian pass (its register sets do not fit), so
        # its three calls are also its fastest step
        ms64, st64 = ms64s, st64s
        extra["fp64_ms_per_step"] = round(ms64, 4)
        extra["fp64_stages"] = stage_roofline(st64, field * 16)
        extra["speedup_vs_fp64_gpu"] = round(ms64 / ms, 3)
        # the stated target: the FP32 step at >= 3x the plain FP64 GPU path;
        # both paths are HBM-bound and FP64 moves twice the bytes, so the
        # ratio is bounded near 2 unless FP32 moves fewer sweeps than FP64
        extra["target_vs_fp64_gpu"] = {"target": 3.0, "measured": round(ms64 / ms, 3), "met": ms64 / ms >= 3.0}
        log(f"errors vs FP64 GPU path: {json.dumps(errs)}")
        # the FP64 path with the reference's stage structure: per direction
        # FFT1a + pack + exchange, then unpack + twiddle + FFT1b, materialising
        # the post-exchange buffer (zmodel/transforms/fft.cu:199-339)
        if not args.two_stage:
            plan64s = Plan(dims, n, p, b, precision="fp64", two_stage=True)
            ms64t, _, outs64s = time_path(plan64s, x64r, n, max(3, min(args.steps, 10)), 2, torch,
                                          "fp64 two-stage", False)
            extra["fp64_two_stage_ms_per_step"] = round(ms64t, 4)
            extra["speedup_vs_fp64_two_stage_gpu"] = round(ms64t / ms, 3)
            del outs64s, plan64s
        # the split-precision MFMA variant of the same step
        if not args.no_mfma and args.precision == "fp32" and not args.two_stage:
            try:
                pm = Plan(dims, n, p, b, precision="fp32_mfma")
            except Exception as e:  # shapes without radix-16 stages have no MFMA variant
                log(f"no fp32_mfma plan for this shape: {e}")
                pm = None
            if pm is not None:
                msm, stm, outsm = time_path(pm, x, n, args.steps, args.warmup, torch, "fp32_mfma", fused)
                errm = compare_outputs(pm, plan64, x, x64r, outsm, outs64, n, torch)
                del outsm
                c, t = stm["line"]
                extra["fp32_mfma"] = {
                    "ms_per_step": round(msm, 4), "gflops": round(flops / (msm * 1e-3) / 1e9, 1),
                    "step_hbm_frac_2sweep": round(bytes_2sweep / (msm * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
                    "speedup_vs_fp64_gpu": round(ms64 / msm, 3),
                    "line_avg_launch_ms": round(t / c, 4),
                    "line_achieved_gbs": round(per_launch / (t / c * 1e-3) / 1e9, 1),
                    "stages": stage_roofline(stm, field * esize),
                    "errors_vs_fp64_gpu": errm,
                }
                log(f"fp32_mfma: {json.dumps(extra['fp32_mfma'])}")
                del pm
        del x64r

    if not args.no_library_fft:
        torch.cuda.empty_cache()
        extra["library_fft"] = library_fft_comparison(plan, x, n, max(3, min(args.steps, 10)), 2, torch)

    cpu = None
    if not args.no_cpu_baseline:
        torch.cuda.empty_cache()
        if outs64 is None:
            _, _, outs64 = time_path(plan64, x.to(torch.complex128), n, 1, 1, torch, "fp64", False)
        # the CPU legs run on the input of the FP64 GPU path: the field as
        # rounded for the timed precision, promoted back to complex128
        nat_in = plan64.packed_to_natural(x.to(torch.complex128)).cpu().numpy()
        cpu = cpu_baseline(nat_in, dims, n, p, b, args.seed, outs64, plan64, torch)
        del nat_in
    del outs, outs64
    torch.cuda.empty_cache()

    if dims == 2 and not args.no_3d and not args.no_fp64 and (n, p, b) == (8192, 4, 32):
        extra["config_3d"] = leg_3d(args, torch, Plan)

    line = {
        "metric": "FFT GFLOP/s (5N·log2N), % HBM BW peak; FP32 vs FP64 path at stated error",
        "value": round(gflops, 2),
        "unit": "GFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f64" if args.precision == "fp64" else "f32",
        "data": "synthetic",
        "config": {
            "workload": (f"{dims}D N={n} P={p} B={b} ({p ** dims} virtual ranks): {5 if dims == 2 else 7}-point "
                         f"Laplacian (h=1/N) -> forward FFT -> inverse FFT (1/N^{dims}), complex "
                         f"{'128' if args.precision == 'fp64' else '64'}"),
            "n": n, "p": p, "b": b, "precision": args.precision,
            "path": "two-stage" if args.two_stage else ("Laplacian fused into the forward x pass" if fused
                                                        else "three calls"),
            "field": field_desc,
        },
        "roofline": roofline,
        "cpu_baseline": cpu,
        **extra,
    }
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
