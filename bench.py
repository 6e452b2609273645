#!/usr/bin/env python3
"""Benchmark of the dispatch / combine hot path on one MI355X.

A step is one cached-handle dispatch followed by one combine of the DeepSeek-V3-shaped batch
(4096 tokens x 7168 bf16, 256 experts, top-8, 10% of choices masked, expanded layout with
zero_padding) through the public API, with every input already resident in HBM.  The script prints
ONE JSON line: whole-step achieved HBM bandwidth (algorithmic bytes / wall time), the per-kernel
microseconds measured with HIP events on the stream the kernels run on, the roofline of the
dominant kernel and a CPU baseline (the torch-CPU oracle timed on this host's cores).

`ms_per_step` and `value` are the region the command line asks for: --warmup untimed steps, then
exactly --steps timed steps between two device synchronisations.  The per-kernel figures (and
`ms_per_step_median_regions`) come from a longer protocol that is the same whatever --steps says: at
least 20 untimed warm-up launches, then REGIONS timed regions of REGION_LAUNCHES back-to-back
launches each, every region bracketed by a device synchronisation and two HIP events on the stream
the results are consumed on; the figure reported for a kernel is the MEDIAN of the regions'
per-launch times, with the fastest region beside it (`*_min`).  Plain streams of the same bytes
(`stream_ceiling`: nanoep_stream_probe launches in the shape of the kernels) are timed in the same
run and every roofline entry carries `frac_of_stream_ceiling` beside `frac`.  The other benchmark
shapes follow under `roofline_by_workload` (same protocol, shorter CPU samples; `--workload
deepseek-v3` leaves them out), a row of figures each; `--record FILE` keeps everything that was measured.
"""

from __future__ import annotations

import argparse
import json
import os
import re
import statistics
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))

HBM_PEAK_GBS = 8000.0  # MI355X published HBM3E peak
WARMUP_MIN = 20        # untimed launches ahead of every series of timed regions
REGIONS = 7            # timed regions per figure
REGION_LAUNCHES = 100  # back-to-back launches per region
HEADLINE = "deepseek-v3"


def log(*parts):
    print(*parts, file=sys.stderr, flush=True)


def parse_args():
    parser = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    parser.add_argument("--gpus", type=int, default=1)
    parser.add_argument("--steps", type=int, default=200)
    parser.add_argument("--warmup", type=int, default=50)
    parser.add_argument("--workload", default="all",
                        help="`all` (default): the headline shape, then the other benchmark shapes under roofline_by_workload; "
                             "or the name of one shape")
    parser.add_argument("--cpu-seconds", type=float, default=15.0, help="CPU baseline budget per workload; 0 skips it")
    parser.add_argument("--no-scalar-oracle", dest="scalar_oracle", action="store_false",
                        help="skip timing the scalar-loop oracle (it runs once on the readme-toy and mixtral shapes only: "
                             "it is a specification, not a performance path)")
    parser.add_argument("--regions", type=int, default=REGIONS)
    parser.add_argument("--region-launches", type=int, default=REGION_LAUNCHES)
    parser.add_argument("--series", choices=["all", "basic", "streams"], default="all",
                        help="`basic`: only fresh dispatches and the cold step / dispatch / combine series (what a profiler run wants: "
                             "every launch of a kernel name is then the same work); `streams`: only the plain streams")
    parser.add_argument("--no-calibration", dest="calibration", action="store_false",
                        help="skip the plain streams (nanoep_stream_probe) that give every roofline entry its frac_of_stream_ceiling")
    parser.add_argument("--record", metavar="FILE", default="",
                        help="also write everything that was measured there, as JSON (the printed line leaves out the plain streams, the switches, "
                             "the graph and side-stream series and the other workloads' details)")
    parser.add_argument("--calibration-copy-mib", type=int, default=0,
                        help="also launch the plain copy kernel on this many MiB (known-size reference for profiler byte counters)")
    return parser.parse_args()


def measured_traffic(kernel: str, workload: str):
    """(HBM bytes per launch, where that number comes from) out of the committed profiler summary.

    The counters are not collected by this run: they come from two `rocprofv3 --pmc` runs of this
    script whose summary is kept under profiles/, and `source` names that file and the commit the
    library was built from when it was taken, so that a stale summary shows."""
    path = ROOT / "profiles" / f"{kernel}_{workload}_pmc.txt"
    if not path.exists():
        return None, None
    text = path.read_text()
    match = re.search(r"^traffic_bytes_per_launch:\s*([0-9.eE+]+)", text, flags=re.M)
    commit = re.search(r"^source_commit:\s*(\S+)", text, flags=re.M)
    source = {"file": str(path.relative_to(ROOT)), "commit": commit.group(1) if commit else "not recorded",
              "collected_by": "rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE (separate runs), not by this run"}
    return (float(match.group(1)) if match else None), source


def layout_gpu_us(workload, idx, iterations=100):
    """GPU time of the routing-layout launches alone (no host wait), through the C ABI."""
    import ctypes

    import torch

    library = ctypes.CDLL(str(ROOT / "nanoep_amd" / "libnanoep_hip.so"))
    p, i64 = ctypes.c_void_p, ctypes.c_int64
    library.nanoep_layout_workspace_bytes.restype = ctypes.c_size_t
    library.nanoep_layout_workspace_bytes.argtypes = [i64, ctypes.c_int, i64]
    library.nanoep_slot_order_entries.restype = i64
    library.nanoep_slot_order_entries.argtypes = [i64, ctypes.c_int, i64]
    library.nanoep_layout.argtypes = [p, i64, ctypes.c_int, i64, i64, ctypes.c_int, ctypes.c_int, p, p, p, p, p, p, p, p, p, p, ctypes.c_size_t, p, p]
    tokens, topk, experts = workload.tokens, workload.topk, workload.experts
    device = idx.device
    nbytes = library.nanoep_layout_workspace_bytes(tokens, topk, experts)
    workspace = torch.empty(nbytes, dtype=torch.uint8, device=device)
    metadata = torch.empty((tokens, topk + 2), dtype=torch.int32, device=device)
    table = torch.empty((tokens, topk), dtype=torch.int32, device=device)
    order = torch.empty(max(1, library.nanoep_slot_order_entries(tokens, topk, experts)), dtype=torch.int64, device=device)
    snapshot = torch.empty_like(idx)
    dst_slots = torch.empty((tokens, 1), dtype=torch.int64, device=device)
    counts = torch.empty(experts, dtype=torch.int64, device=device)
    offsets = torch.empty(experts + 1, dtype=torch.int64, device=device)
    sent = torch.empty(1, dtype=torch.int64, device=device)
    prefix = torch.empty(1, dtype=torch.int64, device=device)
    mailbox = torch.empty(4, dtype=torch.int64, pin_memory=True)
    stream = torch.cuda.current_stream()

    def launch():
        status = library.nanoep_layout(idx.data_ptr(), tokens, topk, experts, workload.alignment, int(workload.expand),
                                       workload.hidden, metadata.data_ptr(), counts.data_ptr(), offsets.data_ptr(), dst_slots.data_ptr(),
                                       sent.data_ptr(), snapshot.data_ptr(), prefix.data_ptr(),
                                       table.data_ptr() if workload.expand else None,
                                       order.data_ptr() if workload.expand else None, workspace.data_ptr(), nbytes,
                                       mailbox.data_ptr(), stream.cuda_stream)
        if status != 0:
            raise RuntimeError(f"nanoep_layout failed with status {status}")

    for _ in range(WARMUP_MIN):
        launch()
    samples = []
    for _ in range(5):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        torch.cuda.synchronize()
        begin.record(stream)
        for _ in range(iterations):
            launch()
        end.record(stream)
        torch.cuda.synchronize()
        samples.append(begin.elapsed_time(end) * 1e3 / iterations)
    return statistics.median(samples)


def host_description():
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as info:
            model = next((line.split(":", 1)[1].strip() for line in info if line.startswith("model name")), model)
    except OSError:
        pass
    return model, os.cpu_count() or 1


def cpu_baseline(workload, x, idx, weights, budget_seconds, gpu_dispatched=None, gpu_combined=None, scalar=False):
    """The vectorised torch-CPU oracle on the same batch: dispatch + combine, bounded in time.

    When the GPU results of the same batch are given, they are compared bit for bit with the
    oracle's (NaN-free synthetic data, so plain bit equality is the bar) and the verdict is returned.
    """
    import torch

    from nanoep_amd import workloads
    from oracle import nanoep_oracle as oracle

    cpu_model, host_cpus = host_description()
    # the GPU box gives one GPU's share of its host: 16 cores, whatever the machine has
    cores = min(16, host_cpus)
    torch.set_num_threads(cores)
    layout = oracle.layout(idx, workload.experts, workload.alignment)
    received, capacity = layout.recv_count, layout.expanded_capacity
    assignments = int(layout.expert_counts.sum())
    nbytes = (workloads.dispatch_bytes(workload, received, assignments, capacity)
              + workloads.combine_bytes(workload, received, assignments, weighted=workload.combine_weights))
    metadata = layout.recv_metadata(workload.expand)

    def step():
        out_x, _, out_w, _ = oracle.dispatch(x, idx, workload.experts, weights, do_expand=workload.expand,
                                             alignment=workload.alignment, lay=layout)
        oracle.combine(out_x, metadata, layout.dst_slots, do_expand=workload.expand,
                       weights=out_w if workload.combine_weights else None)

    parity = None
    if gpu_dispatched is not None:
        want_x, _, want_w, _ = oracle.dispatch(x, idx, workload.experts, weights, do_expand=workload.expand,
                                               alignment=workload.alignment, lay=layout)
        want_combined, _ = oracle.combine(want_x, metadata, layout.dst_slots, do_expand=workload.expand)
        parity = bool(torch.equal(gpu_dispatched.view(torch.int16), want_x.view(torch.int16))
                      and torch.equal(gpu_combined.view(torch.int16), want_combined.view(torch.int16)))
        del want_x, want_combined

    def sample(limit_seconds, limit_steps):
        step()  # warm caches and the allocator
        times = []
        started = time.perf_counter()
        while True:
            t0 = time.perf_counter()
            step()
            times.append(time.perf_counter() - t0)
            if time.perf_counter() - started > limit_seconds or len(times) >= limit_steps:
                break
        return statistics.median(times), len(times)

    seconds, count = sample(budget_seconds, 20)
    torch.set_num_threads(1)
    single_seconds, single_count = sample(budget_seconds / 2, 5)
    torch.set_num_threads(cores)
    baseline = {
        "value": round(nbytes / seconds / 1e9, 3),
        "unit": "GB/s",
        "cores": cores,
        "host_cpu_count": host_cpus,
        "cpu_model": cpu_model,
        "kind": "port",
        "us_per_step": round(seconds * 1e6, 1),
        "value_1_thread": round(nbytes / single_seconds / 1e9, 3),
        "sample": f"{count} timed steps (cached-layout dispatch + combine) of the full {workload.name} batch "
                  f"with the vectorised torch-CPU oracle, {cores} threads; {single_count} steps with 1 thread",
    }
    if scalar and workload.tokens * workload.topk <= 4096 * 2:
        # the scalar-loop restatement of the reference's oracle, once, for the record
        t0 = time.perf_counter()
        out_x, _, _, scalar_layout = oracle.dispatch_scalar(x, idx, workload.experts, weights, do_expand=workload.expand,
                                                            alignment=workload.alignment)
        oracle.combine_scalar(out_x, scalar_layout.recv_metadata(workload.expand), scalar_layout.dst_slots, do_expand=workload.expand)
        elapsed = time.perf_counter() - t0
        baseline["scalar_oracle_us_per_step"] = round(elapsed * 1e6, 1)
        baseline["scalar_oracle_GBps"] = round(nbytes / elapsed / 1e9, 4)
    return baseline, parity


def summarize(samples_seconds, launches):
    """(median, min) microseconds per launch over timed regions of `launches` launches each."""
    per_launch = [s / launches * 1e6 for s in samples_seconds]
    return statistics.median(per_launch), min(per_launch)


_library = None


def kernel_library():
    """ctypes handle of libnanoep_hip.so for the calls that have no Python API: plain streams, tuning
    switches, the calibration copy."""
    global _library
    if _library is None:
        import ctypes

        library = ctypes.CDLL(str(ROOT / "nanoep_amd" / "libnanoep_hip.so"))
        p, i64 = ctypes.c_void_p, ctypes.c_int64
        library.nanoep_stream_probe.argtypes = [ctypes.c_int, p, p, i64, ctypes.c_int, ctypes.c_int, i64, ctypes.c_int, p]
        library.nanoep_set_tuning.argtypes = [ctypes.c_char_p, ctypes.c_int]
        library.nanoep_copy_bytes.argtypes = [p, p, ctypes.c_size_t, p]
        library.nanoep_reset_tuning.restype = None
        _library = library
    return _library


STREAM_WINDOWS = (64, 128, 256, 512)
STREAM_FANS = (1, 2, 4, 7, 8)


def stream_ceilings(workload, received, assignments, capacity, regions, launches):
    """What plain streams of (nearly) the same bytes attain in this run: for the dispatch a fan-out
    (every source row written `fan` times, windows of source rows that fit an XCD's L2), for the
    combine a fan-in, both with one workgroup per destination row and one wavefront per KiB like the
    kernels, no lookups, rotating sources.  The best window is reported.  Compact layouts are 1:1."""
    import torch

    library = kernel_library()
    hidden = workload.hidden
    if hidden > 8192 or received < max(STREAM_WINDOWS):
        return None  # a latency-sized batch has no bandwidth ceiling worth the name
    written = (capacity if workload.zero_padding else assignments) if workload.expand else received
    ratio = written / received
    fan = min(STREAM_FANS, key=lambda f: abs(f - ratio))
    span = max(STREAM_WINDOWS) * fan
    source_rows = max(max(STREAM_WINDOWS), received // max(STREAM_WINDOWS) * max(STREAM_WINDOWS))
    wide_rows = source_rows * fan
    row = 2 * hidden
    device = torch.device("cuda", 0)
    generator = torch.Generator(device=device).manual_seed(3)

    def rotating(rows):
        copies = min(32, max(3, -(-3 * (256 << 20) // (rows * row))))
        return [torch.randn((rows, hidden), device=device, generator=generator, dtype=torch.float32).to(torch.bfloat16) for _ in range(copies)]

    stream = torch.cuda.current_stream()

    def timed_probe(kind, sources, targets, rows, window, waves):
        def launch(i):
            status = library.nanoep_stream_probe(kind, sources[i % len(sources)].data_ptr(), targets[i % len(targets)].data_ptr(), rows,
                                                 hidden, fan, window, waves, stream.cuda_stream)
            if status != 0:
                raise RuntimeError(f"nanoep_stream_probe failed with status {status}")

        for i in range(WARMUP_MIN):
            launch(i)
        samples = []
        for region in range(regions):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            begin.record(stream)
            for i in range(launches):
                launch(region * launches + i)
            end.record(stream)
            torch.cuda.synchronize()
            samples.append(begin.elapsed_time(end) * 1e3 / launches)
        return statistics.median(samples)

    # workgroup shapes tried: a whole row (up to 16 wavefronts), and two or four consecutive KiB
    shapes = sorted({0, 2, 4})

    def best_of(kind, sources, targets, rows, windows):
        tried = {(window, waves): timed_probe(kind, sources, targets, rows, window, waves) for window in windows for waves in shapes}
        (window, waves), us = min(tried.items(), key=lambda item: item[1])
        return {"window": window, "waves_per_workgroup": waves or "row", "us": round(us, 2), "GBps": round(nbytes / us / 1e3, 1),
                "us_by_window_and_workgroup": {f"{w}/{v or 'row'}": round(t, 2) for (w, v), t in tried.items()}}

    nbytes = (source_rows + wide_rows) * row
    result = {"fan": fan, "source_rows": source_rows, "bytes": nbytes, "windows_tried": list(STREAM_WINDOWS)}
    narrow, wide = rotating(source_rows), [torch.empty((wide_rows, hidden), dtype=torch.bfloat16, device=device) for _ in range(3)]
    result["dispatch"] = dict(best_of(2, narrow, wide, wide_rows, STREAM_WINDOWS), kind=f"fan-out 1:{fan}")
    del narrow, wide
    torch.cuda.empty_cache()
    wide, narrow = rotating(wide_rows), [torch.empty((source_rows, hidden), dtype=torch.bfloat16, device=device) for _ in range(3)]
    result["combine"] = dict(best_of(3, wide, narrow, source_rows, STREAM_WINDOWS), kind=f"fan-in {fan}:1")
    del wide, narrow
    torch.cuda.empty_cache()
    # the pure directions, same launch shapes: all of the step's bytes written, all of them read
    total_rows = source_rows + wide_rows
    target = [torch.empty((total_rows, hidden), dtype=torch.bfloat16, device=device)]
    result["fill"] = {key: value for key, value in best_of(1, target, target, total_rows, (1,)).items() if key in ("us", "GBps", "waves_per_workgroup")}
    sources = [target[0], torch.empty_like(target[0]), torch.empty_like(target[0])]
    result["read"] = {key: value for key, value in best_of(0, sources, target, total_rows, (1,)).items() if key in ("us", "GBps", "waves_per_workgroup")}
    del sources, target
    torch.cuda.empty_cache()
    return result


def roofline_entry(kernel, workload_name, nbytes, median_us, min_us, ceiling=None):
    traffic, source = measured_traffic(kernel, workload_name)
    achieved = nbytes / median_us / 1e3
    entry = {
        "kernel": kernel,
        "bound": "hbm",
        "achieved": round(achieved, 1),
        "peak": HBM_PEAK_GBS,
        "unit": "GB/s",
        "frac": round(achieved / HBM_PEAK_GBS, 4),
        "frac_fastest_region": round(nbytes / min_us / 1e3 / HBM_PEAK_GBS, 4),
        "traffic": traffic,
        "traffic_source": source,
        "algorithmic_bytes": nbytes,
        "avg_us": round(median_us, 2),
        "min_us": round(min_us, 2),
    }
    if ceiling is not None:
        entry["stream_ceiling_GBps"] = ceiling["GBps"]
        entry["stream_ceiling"] = f"{ceiling['kind']}, windows of {ceiling['window']} rows, workgroups of {ceiling['waves_per_workgroup']} KiB"
        entry["frac_of_stream_ceiling"] = round(achieved / ceiling["GBps"], 4)
    return entry


def measure_streams(workload, args, device):
    """Only the plain streams of one workload's bytes (`--series streams`)."""
    import torch

    from nanoep_amd import Buffer, EPConfig, workloads

    x_cpu, idx_cpu, w_cpu = workloads.make_inputs(workload, seed=0)
    with Buffer(None, EPConfig(workload.experts, workload.topk, workload.hidden, workload.tokens)) as buffer:
        layout = buffer.dispatch(x_cpu.to(device), topk_idx=idx_cpu.to(device), do_expand=workload.expand,
                                 alignment=workload.alignment).handle.layout
        received, capacity, assignments = layout.recv_count, layout.expanded_capacity, int(layout.expert_counts.sum().item())
    torch.cuda.empty_cache()
    return {"received_rows": received, "assignments": assignments, "expanded_capacity": capacity,
            "timing": {"warmup_launches": WARMUP_MIN, "regions": min(max(1, args.regions), 3), "launches_per_region": min(max(1, args.region_launches), 40)},
            "stream_ceiling": stream_ceilings(workload, received, assignments, capacity, min(max(1, args.regions), 3),
                                              min(max(1, args.region_launches), 40))}


def measure(workload, args, device, detailed):
    """All figures of one workload.  `detailed` adds the layout, seven-tensor-handle and --steps
    figures (the headline workload)."""
    import dataclasses

    import torch

    from nanoep_amd import Buffer, EPConfig, workloads

    # Rotating source copies: at least 8, and at least three times the 256 MiB last-level cache in
    # total, so that no launch finds its source cache resident (14 x 58.7 MB at the headline batch,
    # 24 copies of a 33.5 MB source).  Copy 0 is the batch that is checked against the oracle.
    x_cpu, idx_cpu, w_cpu = workloads.make_inputs(workload, seed=0)
    source_bytes = max(1, x_cpu.numel() * x_cpu.element_size())
    rotation = min(32, max(8, -(-3 * (256 << 20) // source_bytes)))
    generator = torch.Generator(device=device).manual_seed(1)
    xs = [x_cpu.to(device)] + [
        torch.randn(x_cpu.shape, device=device, generator=generator, dtype=torch.float32).to(torch.bfloat16)
        for _ in range(rotation - 1)
    ]
    idx = idx_cpu.to(device)
    weights = w_cpu.to(device)
    regions, launches = max(1, args.regions), max(1, args.region_launches)
    library = kernel_library()

    buffer = Buffer(None, EPConfig(workload.experts, workload.topk, workload.hidden, workload.tokens))
    asynchronous = workload.async_op
    # The loop makes the buffer's communication stream current, so kernels, HIP events and the caller
    # share one queue and a series of back-to-back calls times the kernels' launch period.  A workload
    # with async_op=True is timed a second time below with the caller on a stream of its own that
    # waits on every call's completion event (`side_stream_consumer`).
    stream = buffer.comm_stream
    result = {}
    with torch.cuda.stream(stream):
        # fresh dispatch: layout kernels + host wait for N/C + permute, as seen by the caller
        # (two series: wall clock around call + synchronisation with nothing else in between, then the
        # same calls between two HIP events, whose recording costs the host a few microseconds)
        fresh_times, fresh_gpu_times = [], []
        fresh_calls = WARMUP_MIN + (4 * rotation if detailed else 20)
        for with_events in (False, True):
            for call in range(fresh_calls, -1, -1):  # rotating sources like the timed steps; the last call takes xs[0]
                begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                torch.cuda.synchronize()
                t0 = time.perf_counter()
                if with_events:
                    begin.record(stream)
                received = buffer.dispatch(xs[call % rotation], topk_idx=idx, weights=weights, do_expand=workload.expand,
                                           alignment=workload.alignment, zero_padding=workload.zero_padding)
                if with_events:
                    end.record(stream)
                torch.cuda.synchronize()
                if call < fresh_calls - WARMUP_MIN:
                    if with_events:
                        fresh_gpu_times.append(begin.elapsed_time(end) * 1e-3)
                    else:
                        fresh_times.append(time.perf_counter() - t0)
        handle = received.handle
        check_combined = buffer.combine(received.x, handle).x
        torch.cuda.synchronize()
        gpu_dispatched, gpu_combined = received.x.cpu(), check_combined.cpu()
        held_bytes = received.x.untyped_storage().nbytes()
        del check_combined
        n_recv, capacity = handle.layout.recv_count, handle.layout.expanded_capacity
        assignments = int(handle.layout.expert_counts.sum().item())
        d_bytes = workloads.dispatch_bytes(workload, n_recv, assignments, capacity)
        c_bytes = workloads.combine_bytes(workload, n_recv, assignments, weighted=workload.combine_weights)

        ring = [received.x, received.x.clone(), received.x.clone()]  # combine reads a two-steps-old dispatch output
        ring_weights = received.topk_weights if workload.combine_weights else None
        replayed = {"handle": handle}

        def do_dispatch(i):
            out = buffer.dispatch(xs[i % rotation], weights=weights, handle=replayed["handle"], zero_padding=workload.zero_padding,
                                  async_op=asynchronous)
            if asynchronous:
                out.event.current_stream_wait()
            ring[i % 3] = out.x

        def do_combine(i):
            out = buffer.combine(ring[(i + 1) % 3], handle, weights=ring_weights, async_op=asynchronous)
            if asynchronous:
                out.event.current_stream_wait()
            return out

        def step(i):
            do_dispatch(i)
            return do_combine(i)

        def do_dispatch_hot(i):
            # the same dispatch when its source is still cache resident (one source copy, as when the
            # producer of x ran just before): reported beside the cold figure, never as `value`
            out = buffer.dispatch(xs[0], weights=weights, handle=handle, zero_padding=workload.zero_padding, async_op=asynchronous)
            if asynchronous:
                out.event.current_stream_wait()
            ring[i % 3] = out.x

        def timed(fn, count, first=0):
            """(wall seconds, GPU seconds between two HIP events on the caller's stream) of `count` calls."""
            current = torch.cuda.current_stream()
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            begin.record(current)
            for i in range(first, first + count):
                fn(i)
            end.record(current)
            torch.cuda.synchronize()
            return time.perf_counter() - t0, begin.elapsed_time(end) * 1e-3

        def series(fn):
            """WARMUP_MIN untimed launches, then the timed regions: lists of wall and GPU seconds."""
            timed(fn, WARMUP_MIN)
            samples = [timed(fn, launches, first=r * launches) for r in range(regions)]
            return [s[0] for s in samples], [s[1] for s in samples]

        def call_to_complete(fn, calls=30):
            """Median microseconds from a call to its results being complete, the device idle before."""
            samples = []
            for i in range(WARMUP_MIN + calls):
                torch.cuda.synchronize()
                t0 = time.perf_counter()
                fn(i)
                torch.cuda.synchronize()
                samples.append(time.perf_counter() - t0)
            return statistics.median(samples[WARMUP_MIN:]) * 1e6

        everything = args.series == "all"
        step_wall, step_gpu = series(step)
        cli = None
        if detailed:
            # The region the command line asks for: --warmup untimed steps, then exactly --steps timed.
            # It follows the step series directly: the caching allocator then hands the outputs the
            # same blocks as in that series (a 20-step region measured 163 us a step here and 167 to
            # 173 us behind the fresh-dispatch and seven-tensor sections below, whose larger and
            # shorter-lived allocations leave the outputs in other blocks of device memory).
            timed(step, max(args.warmup, 0))
            cli_wall, cli_gpu = timed(step, max(1, args.steps))
            cli = {"steps": args.steps, "warmup": args.warmup,
                   "ms_per_step": round(cli_wall / max(1, args.steps) * 1e3, 5),
                   "gpu_us_per_step": round(cli_gpu / max(1, args.steps) * 1e6, 2)}
        _, dispatch_gpu = series(do_dispatch)
        _, combine_gpu = series(do_combine)
        _, hot_gpu = series(do_dispatch_hot) if everything else (None, dispatch_gpu)
        # the same two dispatch series with the walk's window-wise source prefetch forced off and on
        # (on is the library's default; off is for callers whose sources sit in the last-level cache)
        prefetch_gpu = {}
        if workload.expand and everything:
            for setting in (0, 1):
                library.nanoep_set_tuning(b"DISPATCH_PREFETCH", setting)
                prefetch_gpu[setting] = (series(do_dispatch)[1], series(do_dispatch_hot)[1])
            library.nanoep_set_tuning(b"DISPATCH_PREFETCH", -1)
        cached_latency = call_to_complete(do_dispatch) if everything else 0.0
        combine_latency = call_to_complete(do_combine) if everything else 0.0
        layout_us = layout_gpu_us(workload, idx) if detailed and everything else 0.0

        seven = None
        if detailed and workload.expand and everything:
            # A caller that keeps more handles alive than the runtime remembers, and only the seven
            # tensors of each: four more fresh dispatches (other routings) make `handle` the fifth
            # oldest, and its replays go through a copy without the private tensors.  The first replay
            # rebuilds them from the handle itself; the timed ones find them cached.
            keep = []
            for seed in range(1, 5):
                other = workloads.make_inputs(workload, seed=seed)[1].to(device)
                keep.append(buffer.dispatch(xs[0], topk_idx=other, weights=weights, do_expand=True, alignment=workload.alignment).handle)
            rebuilds_before = buffer._runtime.rebuilds()
            recalls_before = buffer._runtime.private_recalls()
            replayed["handle"] = dataclasses.replace(handle, token_slots=None, slot_order=None)
            _, seven_gpu = series(do_dispatch)
            seven_us, seven_min = summarize(seven_gpu, launches)
            seven_x = buffer.dispatch(xs[0], weights=weights, handle=replayed["handle"], zero_padding=workload.zero_padding).x
            torch.cuda.synchronize()
            library.nanoep_set_tuning(b"REBUILD_ORDER", 0)
            _, plain_gpu = series(do_dispatch)
            library.nanoep_set_tuning(b"REBUILD_ORDER", -1)
            seven = {
                "dispatch_us_seven_tensor_handle": round(seven_us, 2),
                "dispatch_us_seven_tensor_handle_min": round(seven_min, 2),
                "dispatch_us_seven_tensor_handle_never_rebuilt": round(summarize(plain_gpu, launches)[0], 2),
                "seven_tensor_handle": {"live_handles_behind_it": len(keep), "rebuilds": buffer._runtime.rebuilds() - rebuilds_before,
                                        "recalls": buffer._runtime.private_recalls() - recalls_before,
                                        "same_bytes_as_the_full_handle": bool(torch.equal(seven_x.view(torch.int16).cpu(), gpu_dispatched.view(torch.int16)))},
            }
            replayed["handle"] = handle
            del keep, seven_x

        side = None
        if asynchronous and everything:
            # the caller on a stream of its own: every call makes the communication stream wait for the
            # caller's stream and the caller's stream wait for the call's completion event
            with torch.cuda.stream(torch.cuda.Stream(device=device)):
                side_step = summarize(series(step)[1], launches)
                side_dispatch = summarize(series(do_dispatch)[1], launches)
                side_combine = summarize(series(do_combine)[1], launches)
            side = {"gpu_us_per_step": round(side_step[0], 2), "dispatch_us": round(side_dispatch[0], 2), "dispatch_us_min": round(side_dispatch[1], 2),
                    "combine_us": round(side_combine[0], 2), "combine_us_min": round(side_combine[1], 2),
                    "timed": "HIP events on the caller's stream around back-to-back dispatch -> event.current_stream_wait() calls: two "
                             "cross-stream waits per call on top of the kernel"}

        ceilings = stream_ceilings(workload, n_recv, assignments, capacity, min(regions, 3), min(launches, 40)) if args.calibration and everything else None

        graph_step = None
        if everything and not asynchronous:
            # The cached step recorded once into a HIP graph (two kernel nodes, the combine reading the
            # dispatch's rows) and replayed: one graph launch a step against two API calls a step.
            # A graph's pointers are fixed, so its source is one tensor (cache resident where it fits);
            # the eager figure beside it runs the same two calls on the same tensor.
            try:
                graph = torch.cuda.CUDAGraph()
                torch.cuda.synchronize()
                with torch.cuda.graph(graph):
                    captured = buffer.dispatch(xs[0], weights=weights, handle=handle, zero_padding=workload.zero_padding)
                    captured_out = buffer.combine(captured.x, handle, weights=captured.topk_weights if workload.combine_weights else None)

                def eager_same_source(i):
                    out = buffer.dispatch(xs[0], weights=weights, handle=handle, zero_padding=workload.zero_padding)
                    return buffer.combine(out.x, handle, weights=out.topk_weights if workload.combine_weights else None)

                graph_gpu = series(lambda i: graph.replay())[1]
                eager_gpu = series(eager_same_source)[1]
                graph_latency = call_to_complete(lambda i: graph.replay())
                eager_latency = call_to_complete(eager_same_source)
                graph.replay()
                torch.cuda.synchronize()
                same = bool(torch.equal(captured_out.x.view(torch.int16).cpu(), gpu_combined.view(torch.int16)))
                graph_step = {
                    "gpu_us_per_step": round(summarize(graph_gpu, launches)[0], 2),
                    "eager_gpu_us_per_step": round(summarize(eager_gpu, launches)[0], 2),
                    "us_call_to_complete": round(graph_latency, 1),
                    "eager_us_call_to_complete": round(eager_latency, 1),
                    "same_bytes_as_eager": same,
                    "step": "cached-handle dispatch + combine of its rows, one static source tensor; graph: one replay a step, eager: two API calls a step",
                }
                del graph, captured, captured_out
            except RuntimeError as error:  # a capture the runtime refuses is reported, not fatal to the other figures
                graph_step = {"error": str(error).splitlines()[0][:200]}

    wall_us, wall_us_min = summarize(step_wall, launches)
    gpu_step_us, gpu_step_us_min = summarize(step_gpu, launches)
    d_us, d_us_min = summarize(dispatch_gpu, launches)
    c_us, c_us_min = summarize(combine_gpu, launches)
    hot_us, hot_us_min = summarize(hot_gpu, launches)
    value = (d_bytes + c_bytes) / wall_us / 1e3
    # the kernels the library routes this workload to (names as a kernel trace shows them)
    dispatch_kernel = "dispatch_walk_kernel" if workload.expand else "dispatch_compact_kernel"
    if not workload.expand:
        combine_kernel = "combine_compact_kernel"
    else:
        # (nanoep_combine's rule)
        chunks, topk = -(-workload.hidden // 512), workload.topk
        waves = workload.tokens * chunks / torch.cuda.get_device_properties(0).multi_processor_count
        one_token = topk <= 5 or (topk == 6 and (chunks > 4 or waves < 128)) or waves <= (32 if topk <= 12 else 20 if topk <= 16 else 12)
        combine_kernel = "combine_held_kernel" if not one_token else "combine_few_rows_kernel" if workload.topk <= 8 else "combine_rows_kernel"
    result.update(
        {
            "value": round(value, 1),
            "unit": "GB/s",
            "ms_per_step": round(wall_us * 1e-3, 5),
            "ms_per_step_min": round(wall_us_min * 1e-3, 5),
            "config": {
                "workload": workload.name,
                "description": workload.description,
                "tokens": workload.tokens,
                "hidden": workload.hidden,
                "experts": workload.experts,
                "topk": workload.topk,
                "layout": "expanded" if workload.expand else "compact",
                "alignment": workload.alignment,
                "zero_padding": workload.zero_padding,
                "received_rows": n_recv,
                "assignments": assignments,
                "expanded_capacity": capacity,
                "step": "cached-handle dispatch + combine through Buffer.dispatch / Buffer.combine"
                        + (", async_op=True with the caller waiting on each completion event (caller on the communication stream; "
                           "`side_stream_consumer`: caller on a stream of its own)" if workload.async_op else "")
                        + (", combine returning the weights" if workload.combine_weights else ""),
                "rotating_source_copies": rotation,
            },
            "timing": {"warmup_launches": WARMUP_MIN, "regions": regions, "launches_per_region": launches,
                       "reported": "median over regions of the per-launch time; *_min is the fastest region"},
            "frac_of_hbm_peak": round(value / HBM_PEAK_GBS, 4),
            "gpu_us_per_step": round(gpu_step_us, 2),
            "gpu_us_per_step_min": round(gpu_step_us_min, 2),
            "dispatch_us": round(d_us, 2),
            "dispatch_us_min": round(d_us_min, 2),
            "dispatch_GBps": round(d_bytes / d_us / 1e3, 1),
            "combine_us": round(c_us, 2),
            "combine_us_min": round(c_us_min, 2),
            "combine_GBps": round(c_bytes / c_us / 1e3, 1),
            "dispatch_us_cache_resident_source": round(hot_us, 2),
            "dispatch_us_cache_resident_source_min": round(hot_us_min, 2),
            "fresh_dispatch_us_host": round(statistics.median(fresh_times) * 1e6, 1),
            "fresh_dispatch_us_host_min": round(min(fresh_times) * 1e6, 1),
            "fresh_dispatch_us_gpu": round(statistics.median(fresh_gpu_times) * 1e6, 1),
            "cached_dispatch_us_call_to_complete": round(cached_latency, 1),
            "combine_us_call_to_complete": round(combine_latency, 1),
            "fresh_dispatch_held_bytes_over_used": round(held_bytes / max(1, gpu_dispatched.numel() * 2), 3),
            "dispatch_bytes": d_bytes,
            "combine_bytes": c_bytes,
            "roofline": roofline_entry(dispatch_kernel, workload.name, d_bytes, d_us, d_us_min, ceilings and ceilings["dispatch"]),
            "roofline_combine": roofline_entry(combine_kernel, workload.name, c_bytes, c_us, c_us_min, ceilings and ceilings["combine"]),
        }
    )
    if prefetch_gpu:
        result["dispatch_prefetch_switch"] = {
            name: {"dispatch_us": round(summarize(cold, launches)[0], 2),
                   "dispatch_us_cache_resident_source": round(summarize(hot, launches)[0], 2),
                   "frac": round(d_bytes / summarize(cold, launches)[0] / 1e3 / HBM_PEAK_GBS, 4)}
            for name, (cold, hot) in (("off", prefetch_gpu[0]), ("on", prefetch_gpu[1]))
        }
        result["dispatch_prefetch_switch"]["default"] = "on"
    if side is not None:
        result["side_stream_consumer"] = side
    if ceilings is not None:
        result["stream_ceiling"] = ceilings
    if seven is not None:
        result.update(seven)
    if graph_step is not None:
        result["hip_graph_step"] = graph_step
    if detailed:
        result["cli_region"] = cli
        result["layout_us_gpu_no_host_wait"] = round(layout_us, 2)
    buffer.close()
    del xs, ring, received, handle, replayed
    torch.cuda.empty_cache()
    if args.cpu_seconds > 0:
        result["cpu_baseline"], result["bit_exact_vs_oracle"] = cpu_baseline(
            workload, x_cpu, idx_cpu, w_cpu, args.cpu_seconds if detailed else min(args.cpu_seconds, 6.0),
            gpu_dispatched, gpu_combined, scalar=args.scalar_oracle)
    return result


def brief(result):
    """What the printed line holds of the record: the headline with its rooflines and CPU baseline, one row of figures for
    every other workload.  It stays below 8000 characters, so that whoever keeps the end of the output keeps all of it."""
    line = {key: value for key, value in result.items()
            if key not in ("stream_ceiling", "dispatch_prefetch_switch", "hip_graph_step", "side_stream_consumer", "roofline_by_workload")}
    rows = {}
    for name, entry in result.get("roofline_by_workload", {}).items():
        row = {"step_GBps": entry["value"]}
        for call, roofline in (("dispatch", entry["roofline"]), ("combine", entry["roofline_combine"])):
            row[call] = {"us": entry[f"{call}_us"], "frac": roofline["frac"]}
            if "frac_of_stream_ceiling" in roofline:
                row[call]["frac_of_stream_ceiling"] = roofline["frac_of_stream_ceiling"]
            if roofline["traffic"] is not None:
                row[call]["traffic_over_algorithmic"] = round(roofline["traffic"] / roofline["algorithmic_bytes"], 3)
        for key in ("dispatch_us_cache_resident_source", "fresh_dispatch_us_host", "bit_exact_vs_oracle"):
            if key in entry:
                row[key] = entry[key]
        if "side_stream_consumer" in entry:
            row["side_stream_us"] = [entry["side_stream_consumer"][key] for key in ("dispatch_us", "combine_us")]
        if "cpu_baseline" in entry:
            row["cpu_us_per_step"] = entry["cpu_baseline"]["us_per_step"]
        rows[name] = row
    if rows:
        line["roofline_by_workload"] = rows
    return line


# (the largest batch first: it takes the longest and sits furthest above its target, see main())
OTHER_WORKLOADS = ["ep8-share", "deepseek-v3-a128", "short-rows-1024", "short-rows-512", "qwen3-moe", "mixtral", "latency-256", "readme-toy"]


def main():
    args = parse_args()
    if args.gpus != 1:
        log("bench.py measures one rank on ONE GPU; --gpus", args.gpus, "is not supported (no collectives are part of this path)")
        return 2

    import torch

    from nanoep_amd import workloads

    names = [HEADLINE] + OTHER_WORKLOADS if args.workload == "all" else [args.workload]
    if any(name not in workloads.WORKLOADS for name in names):
        log("unknown workload", args.workload, "choose from", sorted(workloads.WORKLOADS), "or all")
        return 2
    device = torch.device("cuda", 0)
    torch.cuda.set_device(device)

    if args.series == "streams":
        print(json.dumps({name: measure_streams(workloads.WORKLOADS[name], args, device) for name in names}), flush=True)
        return 0
    # The other workloads go first and the headline one last.  A process that starts right after
    # another one has given back tens of GiB of device memory (a test suite, the previous tenant of
    # the machine) runs 2 to 4 % below its own later figures for its first ten to twenty seconds,
    # whatever it allocates and however; what it measures after that is what every later run of the
    # same command measures.
    others = {}
    failed = False
    for name in names[1:]:
        log("workload", name)
        entry = measure(workloads.WORKLOADS[name], args, device, detailed=False)
        failed = failed or entry.get("bit_exact_vs_oracle") is False
        others[name] = {key: entry[key] for key in (
            "value", "unit", "ms_per_step", "dispatch_us", "dispatch_us_min", "combine_us", "combine_us_min",
            "dispatch_us_cache_resident_source", "fresh_dispatch_us_host", "cached_dispatch_us_call_to_complete",
            "combine_us_call_to_complete", "roofline", "roofline_combine", "dispatch_prefetch_switch", "side_stream_consumer", "stream_ceiling", "hip_graph_step",
            "cpu_baseline", "bit_exact_vs_oracle") if key in entry}
        others[name]["config"] = {key: entry["config"][key] for key in (
            "tokens", "hidden", "experts", "topk", "layout", "alignment", "zero_padding", "rotating_source_copies", "step")}
    workload = workloads.WORKLOADS[names[0]]
    if others:
        log("workload", names[0])
    measured = measure(workload, args, device, detailed=True)
    cli = measured["cli_region"]
    step_bytes = measured["dispatch_bytes"] + measured["combine_bytes"]
    result = {
        "metric": "dispatch+combine achieved HBM bandwidth (algorithmic bytes / wall time), "
                  f"{workload.tokens}x{workload.hidden} bf16, {workload.experts} experts top-{workload.topk}",
        # the region the command line asked for: --warmup untimed steps, then exactly --steps timed ones
        "value": round(step_bytes / cli["ms_per_step"] / 1e6, 1),
        "unit": measured.pop("unit"),
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": cli["ms_per_step"],
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "payload_dtype": "bf16",
        "data": "synthetic",
        # the longer protocol: median of the timed regions of back-to-back steps
        "value_median_regions": measured.pop("value"),
        "ms_per_step_median_regions": measured.pop("ms_per_step"),
        "ms_per_step_fastest_region": measured.pop("ms_per_step_min"),
    }
    measured["frac_of_hbm_peak_median_regions"] = measured.pop("frac_of_hbm_peak")
    result["frac_of_hbm_peak"] = round(result["value"] / HBM_PEAK_GBS, 4)
    result.update(measured)
    failed = failed or result.get("bit_exact_vs_oracle") is False
    if others:
        result["roofline_by_workload"] = others
    if args.calibration_copy_mib > 0:
        library = kernel_library()
        nbytes = args.calibration_copy_mib << 20
        source = torch.full((nbytes,), 3, dtype=torch.uint8, device=device)
        target = torch.empty_like(source)
        torch.cuda.synchronize()
        for _ in range(3):
            status = library.nanoep_copy_bytes(source.data_ptr(), target.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream)
            assert status == 0, status
        torch.cuda.synchronize()
        assert torch.equal(source[:4096], target[:4096])
        result["calibration_copy_bytes"] = nbytes
        del source, target
    if failed:
        log("ERROR: GPU results of a timed configuration differ from the oracle")
    if args.record:
        Path(args.record).write_text(json.dumps(result, indent=1) + "\n")
    print(json.dumps(brief(result)), flush=True)
    return 1 if failed else 0


if __name__ == "__main__":
    sys.exit(main())
