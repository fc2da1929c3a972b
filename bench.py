#!/usr/bin/env python3
"""Benchmark of the MI355X tensor-ring operator (driver contract: one JSON line on stdout).

    python bench.py [--gpus 1] [--steps K] [--warmup W]

Workload: y = TR(G1,G2,G3) x, 1920 -> 2880, modes (8,12,20) ->
(12,10,24), rank 8, fp16, tokens = 1, seeded N(0, sigma^2) cores (make_cores, seed 0) and
N(0,1) x (generator seed 0 + T), as the reference harness draws them
(benchmarks/benchmark.py:107-109). A step is one call of the prepared operator; `value` is
its HIP-event stream latency in us/call over exactly K back-to-back calls, bracketed by
synchronizes, with x and the packed cores resident in HBM.

The line (the last line on stdout, kept under LINE_LIMIT bytes) carries the headline, the
dominant kernel's roofline, the CPU baseline (the package's torch restatement of the
reference path and the oracle's port of it, fp32, timed on this host) and one compact row per
metric case (tokens 8/32 at rank 8, 1/32 at rank 16, the bf16 Llama-shaped configs and
config 1 in fp32): stream time, the dense GEMM of the same shape (F.linear on the materialised
weight, timed the same way) and roofline fractions. Kernel-only durations are not measured in
process (every in-process source reads short kernels long); the roofline quotes the committed
rocprofv3 kernel trace of the headline kernel beside its stream figure. The full per-case
records, floors and memory figures go to DETAILS (and a summary line per case to stderr).
Every case is checked against the fp32 factorized path after timing; a result outside the
acceptance tolerance ends the run with a non-zero status and no JSON line.
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
# Kernel arguments in host memory: the HIP runtime's default on this GPU copies them to device
# memory and reads them back before each launch, which costs ~1.5 us of host time per launch
# with arguments (every launch measured here, ours and the dense GEMM alike). Set before HIP
# initialises; an explicit setting in the environment wins.
# `--runtime-default-child` is the child process that times the headline under the runtime's
# own default (the setting unset), reported next to the tuned figure.
if "--runtime-default-child" in sys.argv[1:]:
    os.environ.pop("HIP_FORCE_DEV_KERNARG", None)
else:
    os.environ.setdefault("HIP_FORCE_DEV_KERNARG", "0")
sys.path.insert(0, str(ROOT / "kernel-task_amd"))
sys.path.insert(0, str(ROOT))

METRIC = "µs/call HIP-event latency, tokens 1/8/32, rank 8/16, vs dense fp16 GEMM"
# the run record keeps about the last 10 KB of stdout: the one line stays well inside it
LINE_LIMIT = 8000
DETAILS = ROOT / "gpurun_out" / "bench_details.json"
H100_PUBLISHED_R8_T1_US = 8.18  # the reference's published fused-kernel (ours-B) stream, R8 t1, H100 SXM5

CASES = [  # (label, input modes, output modes, rank, dtype, init, tokens)
    ("r8", (8, 12, 20), (12, 10, 24), 8, "float16", "per_core", (1, 8, 32)),
    ("r16", (8, 12, 20), (12, 10, 24), 16, "float16", "per_core", (1, 32)),
    ("llama_up_r8", (16, 16, 16), (16, 28, 32), 8, "bfloat16", "uniform", (1, 8, 32, 128)),
    ("llama_down_r16", (16, 28, 32), (16, 16, 16), 16, "bfloat16", "uniform", (1, 32, 256)),
    # the reference's CPU-runnable case in fp32 (on fp32 MFMAs), the GPU
    # figure to set beside the CPU baseline, which times the same config
    ("r8_fp32", (8, 12, 20), (12, 10, 24), 8, "float32", "per_core", (1, 8, 32)),
]


def log(msg: str) -> None:
    print(msg, file=sys.stderr, flush=True)


# Acceptance per case (tests/test_correctness.py:17-23 and BASELINE.json north_star): the
# elementwise rule |y - y_ref| <= tol + tol*|y_ref| and, for 16-bit types,
# max|y - y_ref| <= 1e-2 * max|y_ref|.
TOLERANCE = {"float16": 2e-2, "bfloat16": 2e-2, "float32": 1e-4}


def measure_case(label, ins, outs, rank, dtype_name, init, tokens, steps, warmup, headline):
    import torch

    from factorized_inference import (TRSpec, dense_forward, make_cores,
                                      materialize_dense_weight, prepare_optimized,
                                      tr_forward_reference)
    from factorized_inference import measure as m

    dtype = getattr(torch, dtype_name)
    spec = TRSpec(ins, outs, rank)
    cores = make_cores(spec, device="cuda", dtype=dtype, seed=0, init=init)
    m.synchronize()
    mem0 = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    t0 = time.perf_counter()
    run = prepare_optimized(cores, spec)
    m.synchronize()
    prep_ms = (time.perf_counter() - t0) * 1e3
    # device memory: what preparing holds (the packed cores) and its transient peak
    prep_held = torch.cuda.memory_allocated() - mem0
    prep_peak = torch.cuda.max_memory_allocated() - mem0
    weight = materialize_dense_weight(cores, spec)
    results = []
    for T in tokens:
        g = torch.Generator(device="cuda").manual_seed(0 + T)
        x = torch.randn(T, spec.in_features, generator=g, device="cuda", dtype=dtype)
        ours = lambda: run(x)  # noqa: E731
        dense = lambda: dense_forward(x, weight)  # noqa: E731
        one = m.host_us(ours, 1)[0]              # first call; sizes the loops below
        # the headline takes exactly W untimed steps; the other cases warm up for ~0.3 s of
        # calls (the GPU clock takes a few hundred ms of load to settle; 20 calls of a 30 us
        # kernel measured 10 % slow)
        warm = warmup if headline and T == 1 else max(warmup, min(20000, int(0.3e6 / max(one, 1.0))))
        for _ in range(warm):
            ours()
            dense()
        m.synchronize()
        is_head = headline and T == 1
        # other cases: blocks of up to `steps` calls and at most ~0.3 s each (a block of 100
        # calls of a few us lasted under half a millisecond and varied by 10 % between runs)
        calls = steps if is_head else max(5, min(steps, int(0.3e6 / max(one, 1.0))))
        if is_head:
            m.synchronize()                      # barrier + synchronize on both sides
            ours_blocks = m.stream_us(ours, calls, blocks=1)
            m.synchronize()
        else:
            ours_blocks = m.stream_us(ours, calls, blocks=3)
        ours_us = statistics.median(ours_blocks)
        dense_us = statistics.median(m.stream_us(dense, calls, blocks=3))
        host_ours = statistics.median(m.host_us(ours, min(50, calls)))
        host_dense = statistics.median(m.host_us(dense, 50))
        submit_us = m.host_submit_us(ours, min(200, calls))
        # device memory of one call beyond its output (y stays allocated): nothing, no
        # workspace and no counters. Only this case's inputs are alive when the peak is
        # reset (the previous token count's outputs were released at the end of its turn)
        m.synchronize()
        torch.cuda.reset_peak_memory_stats()
        y = run(x)
        m.synchronize()
        call_extra = torch.cuda.max_memory_allocated() - torch.cuda.memory_allocated()
        # correctness after timing, against the fp32 factorized path on the same cores
        yf = y.float()
        ref = tr_forward_reference(x.float(), [c.float() for c in cores], spec)
        diff = (yf - ref).abs()
        err = diff.max().item()
        tol = TOLERANCE[dtype_name]
        ok = bool((diff <= tol + tol * ref.abs()).all().item()) and bool(torch.isfinite(yf).all())
        if dtype_name != "float32":
            ok = ok and err <= 1e-2 * ref.abs().max().item()
        max_ref = ref.abs().max().item()
        del y, yf, ref, diff
        info = run.selected(T)
        flops = run.plan.launch_flops(tokens=T)
        ref_flops = m.reference_flops(spec, T)
        peak = m.PEAK_TFLOPS[dtype]
        case = {
            "case": label, "tokens": T, "rank": rank, "dtype": dtype_name,
            "modes": [list(ins), list(outs)], "variant": info["name"], "grid": info["grid"],
            "lds_bytes": info["lds_bytes"],
            "ours_stream_us": ours_us, "dense_stream_us": dense_us,
            "speedup_vs_dense": dense_us / ours_us,
            "ours_host_us": host_ours, "dense_host_us": host_dense, "ours_submit_us": submit_us,
            "flops": flops, "bytes": info["bytes"],
            "max_abs_err_vs_fp32": err, "max_abs_ref": max_ref,
            "prepare_ms": prep_ms, "packed_bytes": run.packed_bytes,
            "prepare_held_bytes": prep_held, "prepare_peak_bytes": prep_peak,
            "call_extra_bytes": call_extra,
            "dense_weight_bytes": weight.numel() * weight.element_size(),
            "passed": ok,
            **m.roofline(flops, info["bytes"], ours_us, dtype),
            # the reference's flop count (its fixed order) at the same time, for comparison
            # with its "% FP16 TC peak" column
            "reference_flops": ref_flops,
            "frac_mfma_reference_flops": ref_flops / (ours_us * 1e-6) / 1e12 / peak,
        }
        log(f"{label} T={T}: ours {ours_us:.2f} us, dense {dense_us:.2f} us, "
            f"err {err:.2e}{'' if ok else ' FAILED'}, {info['name']}")
        results.append(case)
    return results


def xcd_local_figure(steps: int, warmup: int) -> dict | None:
    """The headline workload on the plan's XCD-local variant (PreparedTRKernel.use_xcd_local:
    every workgroup on one XCD) against the default variant, as a paired comparison: both
    warmed for ~0.3 s, then 9 alternating blocks of `steps` calls each. Checked like every
    case, with the HBM traffic its counter runs measured (profiles/traffic_r8_t1_xl.json)."""
    import torch

    from factorized_inference import TRSpec, make_cores, prepare_optimized, tr_forward_reference
    from factorized_inference import measure as m

    label, ins, outs, rank, dt, init, _ = CASES[0]
    spec = TRSpec(ins, outs, rank)
    cores = make_cores(spec, device="cuda", dtype=torch.float16, seed=0, init=init)
    base = prepare_optimized(cores, spec)
    run = prepare_optimized(cores, spec)
    if not run.use_xcd_local():
        return None
    x = torch.randn(1, spec.in_features, generator=torch.Generator(device="cuda").manual_seed(1),
                    device="cuda", dtype=torch.float16)
    ours = lambda: run(x)  # noqa: E731
    default = lambda: base(x)  # noqa: E731
    t_end = time.perf_counter() + 0.3
    while time.perf_counter() < t_end:
        for _ in range(max(warmup, 50)):
            ours()
            default()
        m.synchronize()
    blocks, default_blocks = [], []
    for _ in range(9):
        blocks += m.stream_us(ours, steps, blocks=1)
        default_blocks += m.stream_us(default, steps, blocks=1)
    y = run(x).float()
    ref = tr_forward_reference(x.float(), [c.float() for c in cores], spec)
    diff = (y - ref).abs()
    tol = TOLERANCE[dt]
    ok = (bool((diff <= tol + tol * ref.abs()).all().item()) and bool(torch.isfinite(y).all())
          and diff.max().item() <= 1e-2 * ref.abs().max().item())
    out = {"variant": run.selected(1)["name"], "value": statistics.median(blocks),
           "default_variant": base.selected(1)["name"],
           "default_value": statistics.median(default_blocks), "unit": "us/call",
           "protocol": f"median of 9 blocks of {steps} calls, alternating with the default",
           "passed": ok, "max_abs_err_vs_fp32": diff.max().item()}
    path = ROOT / "profiles" / "traffic_r8_t1_xl.json"
    if path.exists():
        t = json.loads(path.read_text())
        out.update(traffic=t.get("hbm_bytes_per_launch"), traffic_kernel=t.get("kernel"),
                   traffic_ratio_to_algorithmic=t.get("ratio_to_algorithmic"))
    return out


def cpu_baseline(seconds: float) -> dict:
    """The reference CPU path, config 1 (1920->2880, R8, fp32, T=1, per-core sigma, seed 0),
    timed on this host: the oracle's numpy port of the reference's three contractions
    (`value`, 1 BLAS thread, about `seconds` of work) and, beside it, the package's torch
    restatement of tr_forward_reference (the reference's own CPU path: permute + matmul
    through torch's CPU BLAS) at 1 thread and at every thread count up to the host's."""
    import numpy as np
    import torch
    from threadpoolctl import threadpool_limits

    from factorized_inference import TRSpec, make_cores, tr_forward_reference
    from oracle import ring_oracle

    spec = TRSpec()
    cores_t = make_cores(spec, seed=0)
    cores = [c.numpy() for c in cores_t]
    x_t = torch.randn(1, spec.in_features, generator=torch.Generator().manual_seed(1))
    x = x_t.numpy()

    def sample(fn, budget):
        for _ in range(20):
            fn()
        samples = []
        t_end = time.perf_counter() + budget
        while time.perf_counter() < t_end or len(samples) < 100:
            t0 = time.perf_counter_ns()
            fn()
            samples.append((time.perf_counter_ns() - t0) / 1000.0)
        return statistics.median(samples), len(samples)

    with threadpool_limits(limits=1):
        port_us, port_n = sample(lambda: ring_oracle.tr_forward(x, cores), seconds)
        assert np.isfinite(ring_oracle.tr_forward(x, cores)).all()
    host = os.cpu_count() or 1
    counts = sorted({1, 2, 4, 8, 16, host} & set(range(1, host + 1)))
    before = torch.get_num_threads()
    torch_path = {}
    try:
        with torch.inference_mode():
            for n in counts:
                torch.set_num_threads(n)
                us, calls = sample(lambda: tr_forward_reference(x_t, cores_t, spec),
                                   seconds / 2 if n == 1 else seconds / 8)
                torch_path[str(n)] = {"us": us, "calls": calls}
    finally:
        torch.set_num_threads(before)
    # the baseline is the fastest CPU figure measured (the torch path at its best thread
    # count); the oracle port and every thread count are kept beside it
    best_threads, best = min(torch_path.items(), key=lambda kv: kv[1]["us"])
    return {
        "value": best["us"], "unit": "us/call", "cores": int(best_threads), "kind": "port",
        "sample": (f"config 1 (1920->2880, R8, fp32, T=1, per-core sigma, seed 0): median of "
                   f"{best['calls']} calls of tr_forward_reference on the CPU (the reference's "
                   f"three contractions in its order, torch CPU BLAS, {best_threads} threads)"),
        "torch_reference_path_us": torch_path,
        "oracle_port_us": port_us, "oracle_port_calls": port_n, "oracle_port_threads": 1,
        "host_threads": host, "cpu_model": _cpu_model(),
    }


def _cpu_model() -> str:
    """The host CPU's model name, family and model numbers (/proc/cpuinfo)."""
    fields = {}
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                key, _, value = line.partition(":")
                key = key.strip()
                if key in ("model name", "cpu family", "model", "stepping") and key not in fields:
                    fields[key] = value.strip()
    except OSError:
        return "unknown"
    name = fields.get("model name", "unknown")
    return (f"{name} (family {fields.get('cpu family', '?')}, model {fields.get('model', '?')}, "
            f"stepping {fields.get('stepping', '?')})")


def traffic_probe(calls: int, case: str = "r8:1", variant: str | None = None) -> None:
    """Workload of the rocprofv3 --pmc runs: `calls` launches of one case's kernel (`case` is
    "label:tokens" of CASES; the headline r8:1 by default; `variant` names another compiled
    variant of the plan to launch instead of its default), then a plain 512 MiB device copy
    (5 launches; larger than every L2 and the 256 MB MALL, so its reads come from HBM) whose
    counters give the scale factor between counted and actual bytes."""
    import torch

    from factorized_inference import TRSpec, make_cores, prepare_optimized

    label, _, tok = case.partition(":")
    found = [c for c in CASES if c[0] == label]
    if not found or not tok.isdigit() or int(tok) < 1:
        raise SystemExit(f"--probe-case wants label:tokens with a label of {[c[0] for c in CASES]}")
    _, ins, outs, rank, dt, init, _ = found[0]
    T, dtype = int(tok), getattr(torch, dt)
    spec = TRSpec(ins, outs, rank)
    cores = make_cores(spec, device="cuda", dtype=dtype, seed=0, init=init)
    run = prepare_optimized(cores, spec)
    if variant is not None:
        names = [v["name"] for v in run.variants(T)]
        if variant not in names:
            raise SystemExit(f"--probe-variant {variant!r} is not one of {names}")
        run.plan.set_variant(1, 1 << 30, names.index(variant))
    x = torch.randn(T, spec.in_features, generator=torch.Generator(device="cuda").manual_seed(1),
                    device="cuda", dtype=dtype)
    for _ in range(calls):
        run(x)
    src = torch.ones(256 << 20, dtype=torch.float16, device="cuda")
    dst = torch.empty_like(src)
    for _ in range(5):
        dst.copy_(src)
    torch.cuda.synchronize()
    print(f"traffic probe: {calls} x {run.selected(T)['name']} ({label}, T={T}), 5 x copy of "
          f"{src.numel() * 2} bytes", flush=True)


def runtime_default_child(steps: int, warmup: int) -> int:
    """Child process: the headline measured exactly as in the parent, under the HIP
    runtime's default kernel-argument placement (HIP_FORCE_DEV_KERNARG unset)."""
    import torch

    from factorized_inference import measure as m

    torch.set_num_threads(1)
    with torch.inference_mode():
        a = torch.randn(4096, 4096, device="cuda", dtype=torch.float16)
        t_end = time.perf_counter() + 0.5
        while time.perf_counter() < t_end:
            for _ in range(20):
                a @ a
            torch.cuda.synchronize()
        del a
        label, ins, outs, rank, dt, init, _ = CASES[0]
        case = measure_case(label, ins, outs, rank, dt, init, (1,), steps, warmup,
                            headline=True)[0]
        from factorized_inference import TRSpec, make_cores, prepare_optimized

        spec = TRSpec(ins, outs, rank)
        run = prepare_optimized(make_cores(spec, device="cuda", dtype=torch.float16, seed=0), spec)
        x = torch.randn(1, spec.in_features, generator=torch.Generator(device="cuda").manual_seed(1),
                        device="cuda", dtype=torch.float16)
        blocks = m.stream_us(lambda: run(x), steps, blocks=9)
    print(json.dumps({"value": case["ours_stream_us"], "median_of_9_blocks": statistics.median(blocks),
                      "submit_us": case["ours_submit_us"], "passed": case["passed"],
                      "hip_force_dev_kernarg": os.environ.get("HIP_FORCE_DEV_KERNARG")}), flush=True)
    return 0 if case["passed"] else 1


def runtime_default_figure(steps: int, warmup: int) -> dict | None:
    """Runs runtime_default_child in a fresh process (the setting is read once, when HIP
    initialises) and returns what it printed, or None if it failed."""
    import subprocess

    env = {k: v for k, v in os.environ.items() if k != "HIP_FORCE_DEV_KERNARG"}
    cmd = [sys.executable, str(Path(__file__).resolve()), "--runtime-default-child",
           "--steps", str(steps), "--warmup", str(warmup)]
    try:
        done = subprocess.run(cmd, env=env, capture_output=True, text=True, timeout=300)
    except subprocess.TimeoutExpired:
        log("runtime-default child timed out")
        return None
    if done.returncode != 0:
        log(f"runtime-default child failed ({done.returncode}): {done.stderr[-2000:]}")
        return None
    return json.loads(done.stdout.strip().splitlines()[-1])


def main() -> int:
    ap = argparse.ArgumentParser(description=__doc__.splitlines()[0])
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=400)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--cpu-seconds", type=float, default=10.0)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--headline-only", action="store_true")
    ap.add_argument("--no-runtime-default", action="store_true",
                    help="skip the child process that times the headline under the runtime's "
                         "default kernel-argument placement")
    ap.add_argument("--runtime-default-child", action="store_true", help=argparse.SUPPRESS)
    ap.add_argument("--traffic-probe", type=int, default=0, metavar="CALLS",
                    help="only run the workload of the counter (rocprofv3 --pmc) runs")
    ap.add_argument("--probe-case", default="r8:1", metavar="LABEL:TOKENS",
                    help="case of the --traffic-probe workload (default r8:1, the headline)")
    ap.add_argument("--probe-variant", default=None, metavar="NAME",
                    help="variant the --traffic-probe workload launches (default: the plan's)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU: this build has no multi-GPU path (asked for "
              f"--gpus {args.gpus}); run with --gpus 1", file=sys.stderr)
        return 2
    if args.traffic_probe:
        traffic_probe(args.traffic_probe, args.probe_case, args.probe_variant)
        return 0
    if args.runtime_default_child:
        return runtime_default_child(args.steps, args.warmup)

    import torch

    from factorized_inference import _lib
    from factorized_inference import measure as m

    if not torch.cuda.is_available():
        print("bench.py needs a ROCm GPU", file=sys.stderr)
        return 1
    torch.backends.cuda.matmul.allow_fp16_reduced_precision_reduction = False
    torch.backends.cuda.matmul.allow_bf16_reduced_precision_reduction = False
    torch.set_num_threads(1)
    with torch.inference_mode():
        # bring the GPU to its working clock before the first case (dense GEMMs, untimed)
        a = torch.randn(4096, 4096, device="cuda", dtype=torch.float16)
        t_end = time.perf_counter() + 0.5
        while time.perf_counter() < t_end:
            for _ in range(20):
                a @ a
            torch.cuda.synchronize()
        del a
        cases = []
        for i, (label, ins, outs, rank, dt, init, tokens) in enumerate(CASES):
            if args.headline_only and i > 0:
                break
            cases += measure_case(label, ins, outs, rank, dt, init, tokens, args.steps,
                                  args.warmup, headline=(i == 0))
        floors = m.floors(_lib.load())
        xcd_local = None if args.headline_only else xcd_local_figure(args.steps, args.warmup)
    failed = [f"{c['case']} T={c['tokens']}" for c in cases if not c["passed"]]
    if xcd_local is not None and not xcd_local["passed"]:
        failed.append("r8 T=1 XCD-local")
    if failed:
        log(f"results outside the acceptance tolerance: {', '.join(failed)}; no bench line")
        return 1
    default_runtime = None if args.no_runtime_default else runtime_default_figure(
        args.steps, args.warmup)
    traffic = traffic_figure(cases[0]["variant"])
    cpu = None if args.no_cpu_baseline else cpu_baseline(args.cpu_seconds)
    details = {"cases": cases, "floors": floors, "xcd_local": xcd_local, "cpu_baseline": cpu,
               "runtime_default": default_runtime}
    try:
        DETAILS.parent.mkdir(parents=True, exist_ok=True)
        DETAILS.write_text(json.dumps(details, indent=1) + "\n")
        details_path = str(DETAILS.relative_to(ROOT))
    except OSError as exc:
        log(f"could not write {DETAILS}: {exc}")
        details_path = None
    emit(build_line(args.steps, args.warmup, cases, floors, xcd_local, cpu, default_runtime,
                    traffic, details_path, m.PEAK_HBM_GBS))
    return 0


# per-case row of the line: (column, case key, digits)
CASE_COLUMNS = [
    ("case", "case", None), ("T", "tokens", None), ("ours_us", "ours_stream_us", 2),
    ("dense_us", "dense_stream_us", 2), ("frac_hbm", "frac_hbm", 5),
    ("frac_mfma", "frac_mfma", 4), ("frac_mfma_ref_flops", "frac_mfma_reference_flops", 4),
    ("err", "max_abs_err_vs_fp32", 6),
    ("extra_bytes", "call_extra_bytes", None), ("host_us", "ours_host_us", 1),
    ("variant", "variant", None),
]


def _rounded(v, digits):
    if v is None or digits is None or not isinstance(v, float):
        return v
    return float(f"{v:.{digits}g}") if abs(v) < 1 else round(v, digits)


def trace_kernel_figure(variant: str) -> dict | None:
    """The headline kernel's mean dispatch duration in the committed rocprofv3 kernel trace
    (profiles/ring3_kernel_trace.json, written by benchmarks/counters.py cases from a traced
    run of this script), if that trace is of the same variant."""
    path = ROOT / "profiles" / "ring3_kernel_trace.json"
    try:
        rows = json.loads(path.read_text())["rows"]
    except (OSError, KeyError, ValueError):
        return None
    for r in rows:
        if r.get("variant") == variant and r.get("case") == "r8" and r.get("tokens") == 1:
            return {"mean_us": r["trace_mean_us"], "source": f"rocprofv3 --kernel-trace, "
                    f"{r['trace_dispatches']} dispatches (profiles/ring3_kernel_trace.json)"}
    return None


def traffic_figure(variant: str) -> float | None:
    """HBM bytes per launch of the headline kernel from the committed counter runs
    (profiles/traffic_r8_t1.json, FETCH_SIZE + WRITE_SIZE), if they are of the same variant;
    None otherwise (a default that changed since the counters were taken)."""
    try:
        data = json.loads((ROOT / "profiles" / "traffic_r8_t1.json").read_text())
    except (OSError, ValueError):
        return None
    if f"({variant}:" not in data.get("workload", ""):
        log(f"profiles/traffic_r8_t1.json is of another variant than {variant}: no traffic figure")
        return None
    return data.get("hbm_bytes_per_launch")


def build_line(steps, warmup, cases, floors, xcd_local, cpu, default_runtime, traffic,
               details_path, peak_hbm_gbs) -> dict:
    """The driver's JSON line: headline fields, the dominant kernel's roofline, the CPU
    baseline and a compact row per case (columns CASE_COLUMNS). Long fields (variant names,
    then the runtime-default and XCD-local figures) are dropped if the line would exceed
    LINE_LIMIT bytes; the full records are in the details file."""
    head = cases[0]
    achieved = head["achieved_GBps"]
    roof = {"bound": "hbm", "achieved": achieved, "peak": peak_hbm_gbs, "unit": "GB/s",
            "frac": achieved / peak_hbm_gbs, "traffic": traffic,
            "kernel": head["variant"], "algorithmic_bytes": head["bytes"],
            "time_us": head["ours_stream_us"],
            "time_source": "HIP events (hipEventDisableSystemFence) over the timed block, "
                           "divided by its launches",
            "mfma_frac": head["frac_mfma"],
            "mfma_frac_reference_flops": head["frac_mfma_reference_flops"],
            "floor_stream_empty_args_us": floors.get("stream_empty_launch_args_us"),
            "floor_stream_empty_us": floors.get("stream_empty_launch_us")}
    trace = trace_kernel_figure(head["variant"])
    if trace is not None:
        roof.update({"trace_kernel_us": trace["mean_us"],
                     "trace_kernel_frac": head["bytes"] / (trace["mean_us"] * 1e-6) / 1e9 /
                     peak_hbm_gbs, "trace_source": trace["source"]})
    cpu_short = None
    if cpu is not None:
        cpu_short = {k: cpu[k] for k in ("value", "unit", "cores", "kind", "sample",
                                         "oracle_port_us", "host_threads", "cpu_model")}
        cpu_short["torch_path_us_by_threads"] = {
            n: round(v["us"], 1) for n, v in cpu["torch_reference_path_us"].items()}
    runtime = None
    if default_runtime is not None:
        runtime = {k: default_runtime.get(k) for k in ("value", "median_of_9_blocks", "submit_us")}
    xcd = None
    if xcd_local is not None:
        xcd = {k: xcd_local.get(k) for k in ("variant", "value", "default_value", "traffic")}
    line = {
        "metric": METRIC,
        "value": head["ours_stream_us"],
        "unit": "us/call",
        "n_gpus": 1,
        "steps": steps,
        "warmup": warmup,
        "ms_per_step": head["ours_stream_us"] / 1000.0,
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": head["ours_stream_us"] / H100_PUBLISHED_R8_T1_US,
        "vs_baseline_ref": "reference fused kernel (ours-B) stream, R8 t1, H100 SXM5, 8.18 us (published)",
        "dtype": "f16",
        "data": "synthetic",
        "config": {"workload": "tensor-ring linear 1920->2880, modes (8,12,20)->(12,10,24), "
                               "rank 8, fp16, tokens 1 (BASELINE configs[1])",
                   "tokens": 1, "rank": 8, "in_features": 1920, "out_features": 2880,
                   "hip_force_dev_kernarg": os.environ.get("HIP_FORCE_DEV_KERNARG"),
                   "runtime_default": runtime},
        "dense_stream_us": head["dense_stream_us"],
        "host_us": head["ours_host_us"],
        # preparation of the headline operator (packing the cores into the plan's layout)
        "prepare": {"ms": head["prepare_ms"], "packed_bytes": head["packed_bytes"],
                    "held_bytes": head["prepare_held_bytes"],
                    "peak_bytes": head["prepare_peak_bytes"],
                    "dense_weight_bytes": head["dense_weight_bytes"]},
        "roofline": roof,
        "cpu_baseline": cpu_short,
        "xcd_local": xcd,
        "case_columns": [c for c, _, _ in CASE_COLUMNS],
        "cases": [[_rounded(c.get(k), d) for _, k, d in CASE_COLUMNS] for c in cases],
        "details": details_path,
    }
    if len(json.dumps(line)) > LINE_LIMIT:
        line["case_columns"] = line["case_columns"][:-1]
        line["cases"] = [row[:-1] for row in line["cases"]]
    for key in ("xcd_local", "details"):
        if len(json.dumps(line)) > LINE_LIMIT:
            line.pop(key)
    if len(json.dumps(line)) > LINE_LIMIT:
        line["config"]["runtime_default"] = None
    return line


def emit(line: dict) -> None:
    """Prints the line as the last thing on stdout (everything else goes to stderr)."""
    sys.stdout.flush()
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    sys.exit(main())
