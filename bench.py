#!/usr/bin/env python3
"""Headline benchmark of the serving hot path on one MI355X: requests/s at a p99 latency SLO under mixed-model
Poisson load.

Workload at N=1 (the third benchmark configuration, the one the target statement is about): small CNN (1x1x28x28) and
Inception-v3 (1x3x299x299) at a 9 : 1 request ratio, batch 1, fp32, seeded weights, synthetic inputs; open-loop Poisson
arrivals (exponential inter-arrival times, the arithmetic of reference app/client.cpp:123-212); every request's input
crosses PCIe (host-to-device copy per request, as reference jobs/tvm_mnist/tvm_mnist.cpp:38 does) and its output comes
back; full3 scheduler behind the client library and the shared-memory rings.

SLO: for every tenant, p99 latency (completion minus SCHEDULED arrival) <= SLO_FACTOR x that tenant's latency when it is
served alone with one request outstanding (measured in the same run).  `value` is the highest offered rate, found by
bisection between 0 and the closed-loop saturation rate, at which the SLO holds for both tenants and the served rate
keeps up with the offered one -- re-measured in a final timed run, which is the number reported.

A "step" is a block of STEP_REQUESTS requests of that final run: W warm-up steps are served untimed at the same
offered rate, then exactly K steps are timed from the first submission to the last completion; value = K x
STEP_REQUESTS / elapsed and ms_per_step = elapsed / K.

Beside it, in the same run: the same search for plain multi-stream serving (job-by-job `fifo` on a stream pool, HIP
launches) and for the direct no-server multi-stream loop (reference tests/simple/tvm_direct_multistream.cpp); all arms
at one equal offered load with per-tenant p50/p99 (full3 on direct dispatch, full3 on HIP launches, fifo2, fifo, direct
multi-stream); the other benchmark configurations as side keys; the roofline of the dominant kernel (MFMA implicit-GEMM
conv over Inception-v3's conv launches, per-launch device time stamps), the GPU->host notification probes, the fairness
sweep and the CPU oracle timed on the host cores.

Prints ONE JSON line on stdout; progress goes to stderr.
"""
import argparse
import ctypes
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "requests/sec at p99 latency SLO (mixed-model Poisson load, 1 GPU); notify latency µs"
FP32_MFMA_PEAK_TFLOPS = 157.3
STEP_REQUESTS = 2048      # requests per step of the timed run
SEARCH_REQUESTS = 10240   # requests per point of the rate search
SLO_FACTOR = 10.0         # per-tenant p99 bound, in units of the tenant's alone latency
KEEP_UP = 0.95            # served rate / offered rate below which a point does not count as sustained

# The headline mix and its client-side pools (instances per tenant; the global cap is their sum).
MIX = [("small_cnn", "tvm_mnist", "mnist", 0.9, 96), ("inception_v3", "tvm_inception_v3", "inception_v3", 0.1, 16)]


SUMMARY = []  # the top-level progress lines, printed once more after the detail dump so that they end the stderr stream


def log(*a):
    print(*a, file=sys.stderr, flush=True)
    if len(a) == 1 and isinstance(a[0], str) and a[0].startswith("[bench] ") and not a[0].startswith("[bench]  ") and not a[0].startswith("[bench] detail"):
        SUMMARY.append(a[0])


# HBM-side bytes per conv launch (mean over the conv launches of one forward pass), from FETCH_SIZE / WRITE_SIZE
# counter passes of `bench.py --counter-pass MODEL` scaled by the copy-kernel calibration (FETCH_SIZE x 2.0,
# WRITE_SIZE x 1.0); counters cannot be collected from inside this process, so the figures are carried here.
CONV_TRAFFIC_BYTES_PER_LAUNCH = {"inception_v3": 8.53e6, "resnet18": 6.99e6, "resnet50": 7.10e6, "mobilenetv2": 1.84e6}


def under_counter_collection():
    """True under `rocprofv3 --pmc ...` (it exports its counter list to the profiled process)."""
    return bool(os.environ.get("ROCPROF_COUNTERS"))


def conv_roofline(models, hip, model, reps, back_to_back=200):
    """Per-launch durations of every stage of one forward pass, measured with HIP events on the launch stream."""
    ex = models.Exec(model, seed=1)
    stream = ctypes.c_void_p()
    hip.llis_hip_stream_create(ctypes.byref(stream))
    n = ex.num_stages
    ops = models._abi.ops()
    ev = []
    for _ in range(2):
        e = ctypes.c_void_p()
        hip.llis_hip_event_create(ctypes.byref(e))
        ev.append(e)
    work = [ex.stage_work(i) for i in range(n)]
    for _ in range(3):
        ex.forward(stream)
        hip.llis_hip_stream_synchronize(stream)
    # Each launch stamps the event pair with the kernel's own begin/end time on the device (what a kernel trace
    # reports); one launch at a time on an otherwise idle GPU, in forward-pass order so caches see the real sequence.
    total = [0.0] * n
    ops.paella_ops_time_launches(ev[0], ev[1])
    for _ in range(reps):
        for i in range(n):
            ex.launch_stage(i, stream)
            hip.llis_hip_stream_synchronize(stream)
            ms = ctypes.c_float()
            hip.llis_hip_event_elapsed_ms(ev[0], ev[1], ctypes.byref(ms))
            total[i] += ms.value
    ops.paella_ops_time_launches(None, None)
    per_stage = [t / reps * 1e3 for t in total]  # us
    # back-to-back forward without events: single-stream direct serving rate
    direct_rps = None
    if back_to_back:
        t0 = time.perf_counter()
        for _ in range(back_to_back):
            ex.forward(stream)
        hip.llis_hip_stream_synchronize(stream)
        direct_rps = back_to_back / (time.perf_counter() - t0)
    for e in ev:
        hip.llis_hip_event_destroy(e)
    hip.llis_hip_stream_destroy(stream)
    ex.close()
    conv_flops = sum(w[1] for w in work if w[0] == "conv")
    conv_us = sum(t for t, w in zip(per_stage, work) if w[0] == "conv")
    conv_launches = sum(1 for w in work if w[0] == "conv")
    by_op = {}
    for t, w in zip(per_stage, work):
        d = by_op.setdefault(w[0], {"launches": 0, "us": 0.0, "flops": 0.0, "bytes": 0.0})
        d["launches"] += 1
        d["us"] += t
        d["flops"] += w[1]
        d["bytes"] += w[2]
    return {"per_stage_us": per_stage, "work": work, "conv_flops": conv_flops, "conv_us": conv_us, "conv_launches": conv_launches,
            "by_op": by_op, "direct_rps": direct_rps, "forward_us": sum(per_stage)}


def full_device_pass(models, hip, model, images=16, reps=10, timed=True, kw=None, depth=0, only=None, burst=8, transform=False, one_tile=False):
    """The conv kernel with the device full: every distinct conv layer of the model (groups == 1) over `images` inputs stacked
    along the height, i.e. with `images` times the pixel tiles -- what the compute units see on the serving path, where packed
    launches on four queues keep 16 to 24 problems in flight -- on the 32 x 32 tile with the layer's own waves per workgroup and
    no split of the reduction over workgroups, one launch at a time on a HIP stream.  The library chooses the workgroups: of two tiles,
    as served launches have from 768 on, or of one; one_tile (and kw, depth, transform, which have no other form): of one throughout.  timed: durations from the kernel's own
    begin and end stamps, of the last of `burst` launches enqueued back to back (stream order: they do not overlap; the ones in
    front keep the device's clocks from dropping in the idle gap that a synchronize per launch leaves); otherwise one launch per
    layer with a synchronize after each (for counter collection)."""
    import numpy as np
    import torch
    from paella_amd import ops
    desc = models.describe(model)
    lib = models._abi.ops()
    stream = ctypes.c_void_p()
    hip.llis_hip_stream_create(ctypes.byref(stream))
    ev = []
    for _ in range(2):
        e = ctypes.c_void_p()
        hip.llis_hip_event_create(ctypes.byref(e))
        ev.append(e)
    rng = np.random.default_rng(1)
    seen, rows = {}, []
    for node in desc["nodes"]:
        if node["op"] != "conv" or node["groups"] != 1:
            continue
        x = node["x"]
        key = (x["C"], x["H"], x["W"], node["K"], node["R"], node["S"], tuple(node["stride"]), tuple(node["pad"]))
        if key in seen:
            rows[seen[key]]["count"] += 1
            continue
        c, h, w, k, r, q = x["C"], x["H"], x["W"], node["K"], node["R"], node["S"]
        wt = (rng.standard_normal((k, c, r, q)) / np.sqrt(c * r * q)).astype(np.float32)
        alone = ops.Conv2d(wt, None, stride=tuple(node["stride"]), pad=tuple(node["pad"]), dil=tuple(node["dil"]), act=ops.ACT_RELU, in_hw=(h, w))
        if only and not any(o in "%dx%d %d->%d %dx%d" % (h, w, c, k, r, q) for o in only):
            continue
        # forced shape: waves per workgroup (the layer's own unless given) and chunks of operands in flight per wave (0: default)
        use_kw = kw if kw and c % 8 == 0 else alone.plan.kw
        use_depth = depth if c % 8 == 0 else 0
        hint = (use_depth << 16) | (1 << 8) | (1 << 4) | (use_kw.bit_length() - 1) | (0 if one_tile or kw or depth or transform else 1 << 20)
        conv = ops.Conv2d(wt, np.zeros(k, np.float32), stride=tuple(node["stride"]), pad=tuple(node["pad"]), dil=tuple(node["dil"]), act=ops.ACT_RELU,
                          in_hw=(h * images, w), tile_hint=hint)
        xin = torch.randn((1, c, h * images, w), device="cuda:0")
        y = torch.empty((1, k, conv.plan.P, conv.plan.Q), device="cuda:0")
        # transform: every layer that can apply a per-channel scale-shift to its input on the way does (batch-norm in front of a conv)
        extra = {}
        if transform and conv.takes_input_transform():
            extra = {"in_scale": torch.rand(c, device="cuda:0") + 0.5, "in_shift": torch.randn(c, device="cuda:0")}
        torch.cuda.synchronize()  # the operands are written on torch's stream, the launches go to another
        conv(xin, out=y, stream=stream.value, **extra)
        hip.llis_hip_stream_synchronize(stream)
        us = None
        if timed:
            lib.paella_ops_time_launches(ev[0], ev[1])
            total = 0.0
            for _ in range(reps):
                for _ in range(max(1, burst)):
                    conv(xin, out=y, stream=stream.value, **extra)
                hip.llis_hip_stream_synchronize(stream)
                ms = ctypes.c_float()
                hip.llis_hip_event_elapsed_ms(ev[0], ev[1], ctypes.byref(ms))
                total += ms.value
            lib.paella_ops_time_launches(None, None)
            us = total / reps * 1e3
        seen[key] = len(rows)
        rows.append({"layer": "%dx%d %d->%d %dx%d s%d" % (h, w, c, k, r, q, node["stride"][0]), "count": 1, "workgroups": conv.plan.dims.grid,
                     "waves_per_workgroup": conv.plan.kw, "k_order": conv.plan.k_order, "flops": conv.plan.flops, "us": us,
                     "input_transformed": bool(extra)})
    for e in ev:
        hip.llis_hip_event_destroy(e)
    hip.llis_hip_stream_destroy(stream)
    out = {"model": model, "images": images, "layers": rows}
    if timed:
        # weighted by how often a layer shape occurs in one forward pass
        flops = sum(r["flops"] * r["count"] for r in rows)
        us = sum(r["us"] * r["count"] for r in rows)
        out.update({"achieved": flops / us / 1e6, "frac": flops / us / 1e6 / FP32_MFMA_PEAK_TFLOPS, "unit": "TFLOP/s",
                    "how": "every conv layer of %s over %d inputs stacked along the height (%d times the pixel tiles), 32 x 32 tile, workgroups of %s, one launch at a time "
                           "(the last of %d enqueued back to back); layers weighted by their count in a forward pass" %
                           (model, images, images, "one tile" if one_tile or kw or depth or transform else "two tiles or one as the library chooses",
                            max(1, burst))})
    return out


def multi_queue_rate(models, model, nq=4, reps=200):
    """Forward passes per second with nq requests in flight and no scheduler in between: nq executors, each on its own
    ordered direct-dispatch queue, kernels without hooks.  The GPU-side ceiling of the served path.  Four queues is
    the best this device does: 1/2/3/4/5/6 queues gave 6.2/10.2/13.0/14.5/7.4/8.7 thousand ResNet-18 passes per second."""
    from paella_amd import ops
    execs = [models.Exec(model, seed=1) for _ in range(nq)]
    queues = [ops.DirectQueue(ordered=True) for _ in range(nq)]
    try:
        for e, q in zip(execs, queues):
            e.forward(q.handle)
        for q in queues:
            q.wait()
        t0 = time.perf_counter()
        for _ in range(reps):
            for e, q in zip(execs, queues):
                e.forward(q.handle)
        for q in queues:
            q.wait()
        return nq * reps / (time.perf_counter() - t0)
    finally:
        for q in queues:
            q.close()
        for e in execs:
            e.close()


def cpu_baseline(model, budget_s, max_passes=64):
    from oracle import models as om
    from oracle import ops as orc
    from paella_amd import models
    desc = models.describe(model)
    x = om.make_input(desc, 1)
    om.run(desc, x, seed=1, fast=True)  # touch everything once
    n, t0 = 0, time.perf_counter()
    while True:
        om.run(desc, x, seed=1, fast=True)
        n += 1
        dt = time.perf_counter() - t0
        if dt >= budget_s or n >= max_passes:
            break
    return {"value": n / dt, "unit": "requests/s", "cores": orc.num_threads(), "kind": "port",
            "sample": "%d %s passes in %.1f s" % (n, model, dt)}


def torch_cpu_baseline(model, budget_s):
    """The same graph and seeded weights through torch's CPU operators (oneDNN), all host threads: the stronger CPU
    figure, standing in for the reference's TVM-llvm target, which cannot exist offline."""
    import numpy as np
    import torch
    import torch.nn.functional as F
    from oracle import models as om
    from paella_amd import models
    d = models.describe(model)
    desc = om.Desc(d)
    W = {i: torch.from_numpy(desc.weight(i, 1)) for i in range(len(d["weights"]))}
    bufs = [torch.zeros(b["C"] * b["H"] * b["W"]) for b in d["buffers"]]

    def get(v):
        return None if v["buf"] < 0 else bufs[v["buf"]][v["off"]:v["off"] + v["C"] * v["H"] * v["W"]].view(1, v["C"], v["H"], v["W"])

    def act(y, n):
        a = n["act"]
        if a == 1:
            return F.relu(y)
        if a == 2:
            return torch.clamp(y, 0.0, 6.0)
        if a == 3:
            return F.prelu(y, W[n["slope"]])
        if a == 4:
            return torch.clamp(y, n["lo"], n["hi"])
        return y

    def forward(x):
        get(d["input"]).copy_(x)
        for n in d["nodes"]:
            xin, x2, op = get(n["x"]), get(n["x2"]), n["op"]
            if op == "conv":
                y = F.conv2d(xin, W[n["w"]], W[n["bias"]] if n["bias"] >= 0 else None, tuple(n["stride"]), tuple(n["pad"]), tuple(n["dil"]), n["groups"])
                y = act(y + x2 if x2 is not None else y, n)
            elif op == "dense":
                y = act(F.linear(xin.reshape(1, -1), W[n["w"]], W[n["bias"]]), n)
            elif op == "pool":
                if n["avg"]:
                    y = F.avg_pool2d(xin, tuple(n["k"]), tuple(n["stride"]), tuple(n["pad"]), bool(n["ceil"]), bool(n["count_include_pad"]))
                else:
                    y = F.max_pool2d(xin, tuple(n["k"]), tuple(n["stride"]), tuple(n["pad"]), 1, bool(n["ceil"]))
            elif op == "gap":
                y = xin.mean((2, 3), keepdim=True)
            elif op == "eltwise":
                y = xin
                if n["scale"] >= 0:
                    y = y * W[n["scale"]].view(1, -1, 1, 1)
                if n["shift"] >= 0:
                    y = y + W[n["shift"]].view(1, -1, 1, 1)
                y = act(y + x2 if x2 is not None else y, n)
            elif op == "softmax":
                y = F.softmax(xin.reshape(n["rows"], n["cols"]), 1)
            elif op == "lrn":
                y = F.local_response_norm(xin, n["size"], n["alpha"], n["beta"], n["k"])
            else:
                raise ValueError(op)
            get(n["y"]).copy_(y.reshape(get(n["y"]).shape))
        return get(d["output"]).reshape(-1).clone()

    x = torch.from_numpy(om.make_input(d, 1))
    with torch.no_grad():
        out = forward(x)
        ref = om.run(desc, x.numpy(), seed=1, fast=True)
        if not np.allclose(out.numpy(), ref, rtol=1e-2, atol=1e-3):
            return None  # not the same computation: do not report a time for it
        n, t0 = 0, time.perf_counter()
        while True:
            forward(x)
            n += 1
            dt = time.perf_counter() - t0
            if dt >= budget_s or n >= 2000:
                break
    return {"value": n / dt, "unit": "requests/s", "cores": torch.get_num_threads(), "kind": "port",
            "sample": "%d %s passes in %.1f s" % (n, model, dt)}


class Arm:
    """One way of serving the mix: a scheduler behind the server (with a launch path for the model kernels), or the
    direct no-server multi-stream loop.  run() serves `n` requests at mean inter-arrival `iat_us` (0 = saturation)."""

    verify = 4          # seeded inputs per tenant; every completion is compared with the idle server's answer for its input
    verified = 0        # completions checked so far, over every arm and run of this process
    mismatches = 0

    def __init__(self, serve, label, sched, dispatch, streams, tenants, extra_kernels, unfair=1e6):
        self.serve, self.label, self.sched, self.dispatch, self.streams = serve, label, sched, dispatch, streams
        self.tenants, self.extra_kernels, self.unfair = tenants, extra_kernels, unfair
        self.cap = sum(t[4] for t in tenants)
        self.srv = None

    def __enter__(self):
        if self.sched != "direct":
            os.environ["PAELLA_DISPATCH"] = self.dispatch
            name = "bench%d_%s_%d" % (os.getpid(), self.sched, int(time.time() * 1000) % 100000)
            self.srv = self.serve.Server(name, self.sched, num_streams=self.streams, cpu=4, extra_kernels=self.extra_kernels, unfair=self.unfair)
            self.srv.__enter__()
        return self

    def __exit__(self, *exc):
        if self.srv is not None:
            self.srv.stop()
            self.srv = None
        os.environ.pop("PAELLA_DISPATCH", None)
        return False

    def run(self, iat_us, n, warmup, seed=1, verify=None):
        verify = Arm.verify if verify is None else verify
        if self.sched == "direct":
            r = self.serve.direct_multistream([(t[2], t[3], t[4]) for t in self.tenants], iat_us, self.cap, n, warmup_jobs=warmup, seed=seed,
                                              pin_threads=True)
        else:
            jobs = [(self.serve.job_path(t[1]), t[3], t[4]) for t in self.tenants]
            r = self.serve.client_run(self.srv.name, jobs, iat_us, self.cap, n, warmup_jobs=warmup, seed=seed, pin_threads=True, verify=verify)
            if verify:
                Arm.verified += r["verified_requests"]
                Arm.mismatches += r["mismatches"]
                if r["mismatches"]:
                    log("[bench] %s: %d of %d checked completions DIFFER from the idle server's answer" % (self.label, r["mismatches"], r["verified_requests"]))
        return r


def point_of(r, tenants, offered_rps):
    p = {"offered_rps": offered_rps, "achieved_rps": r["throughput_rps"], "p50_us": r["all"]["p50"], "p99_us": r["all"]["p99"]}
    for k, t in enumerate(tenants):
        p[t[0] + "_p50_us"] = r["per_type"][k]["p50"]
        p[t[0] + "_p99_us"] = r["per_type"][k]["p99"]
        p[t[0] + "_count"] = r["per_type"][k]["count"]
    return p


def meets(point, tenants, slo_us):
    if point["offered_rps"] and point["achieved_rps"] < KEEP_UP * point["offered_rps"]:
        return False
    return all(point[t[0] + "_p99_us"] <= slo_us[t[0]] for t in tenants)


def search_rate(arm, tenants, slo_us, iters=7):
    """Highest offered rate (open-loop Poisson) at which every tenant's p99 meets its SLO and the served rate keeps up:
    closed-loop saturation first, then bisection on the fraction of it.  A point that misses is measured a second time with
    another arrival seed before it counts as a miss (one stall of a host thread is enough to spoil the p99 of a 10 000-request
    point).  Returns (rate or None, saturation, points)."""
    sat = arm.run(0.0, SEARCH_REQUESTS, 512)["throughput_rps"]
    points, lo, hi = [], 0.0, 1.0
    f = 0.5
    for _ in range(iters):
        rate = f * sat
        # 10 240 requests per point, fewer only where they would take more than 1.5 s to arrive (arms whose knee is at a few
        # hundred requests/s), never under 2048
        n_point = min(SEARCH_REQUESTS, max(2048, int(rate * 1.5)))
        for attempt, seed in enumerate((1, 2)):
            p = point_of(arm.run(1e6 / rate, n_point, 512, seed=seed), tenants, rate)
            p["meets_slo"] = meets(p, tenants, slo_us)
            p["attempt"] = attempt
            points.append(p)
            log("[bench]     %-22s offered %8.0f req/s: served %8.0f, p99 %s -> %s" %
                (arm.label, rate, p["achieved_rps"], " / ".join("%.0f" % p[t[0] + "_p99_us"] for t in tenants), "ok" if p["meets_slo"] else "miss"))
            if p["meets_slo"] or p["achieved_rps"] < KEEP_UP * rate:
                break  # met, or plainly beyond what can be served: no second look
        if p["meets_slo"]:
            lo = f
        else:
            hi = f
        f = (lo + hi) / 2
    return (lo * sat if lo > 0 else None), sat, points


def alone_latency(serve, adapter, in_floats, out_floats, n, extra_kernels, streams):
    """Latency of one tenant served alone, one request outstanding (input and output crossing PCIe): the unit of its SLO."""
    import numpy as np
    x = np.random.default_rng(1).random(in_floats, dtype=np.float32)
    name = "bench%d_alone_%d" % (os.getpid(), int(time.time() * 1000) % 100000)
    with serve.Server(name, "full3", num_streams=streams, cpu=4, extra_kernels=extra_kernels) as srv:
        serve.client_single(srv.name, serve.job_path(adapter), x, out_floats, n=max(20, n // 10))
        _, lat = serve.client_single(srv.name, serve.job_path(adapter), x, out_floats, n=n)
    lat = np.sort(lat)
    return {"mean_us": float(lat.mean()), "p50_us": float(lat[len(lat) // 2]), "p99_us": float(lat[int(len(lat) * 0.99)]), "requests": n}


def roofline_of(rl, model):
    achieved = rl["conv_flops"] / (rl["conv_us"] * 1e-6) / 1e12
    return {"bound": "mfma", "achieved": achieved, "peak": FP32_MFMA_PEAK_TFLOPS, "unit": "TFLOP/s", "frac": achieved / FP32_MFMA_PEAK_TFLOPS,
            "traffic": CONV_TRAFFIC_BYTES_PER_LAUNCH.get(model),
            "kernel": "conv_mfma_kernel, conv_small_kernel, conv_tall_kernel and their grouped forms (all %d conv launches of one %s forward pass, one at a time on an idle device)" % (rl["conv_launches"], model),
            "flops_per_launch_avg": rl["conv_flops"] / rl["conv_launches"], "us_per_launch_avg": rl["conv_us"] / rl["conv_launches"],
            "algorithmic_bytes_per_launch_avg": rl["by_op"]["conv"]["bytes"] / rl["conv_launches"]}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20, help="timed steps of %d requests each" % STEP_REQUESTS)
    ap.add_argument("--warmup", type=int, default=2, help="untimed steps served first at the same offered rate")
    ap.add_argument("--num-streams", type=int, default=128)
    ap.add_argument("--cpu-seconds", type=float, default=12.0)
    ap.add_argument("--extra-kernels", type=int, default=48, help="full3: kernels admitted beyond the occupancy budget")
    ap.add_argument("--unfair", type=float, default=1e6, help="full3: deficit threshold of the headline arm (1e6 = shortest remaining work first only)")
    ap.add_argument("--no-arms", action="store_true", help="only the headline search and timed run (plus roofline and CPU baseline)")
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-verify", action="store_true", help="do not compare every completion with the idle server's answer for its input")
    ap.add_argument("--no-side", action="store_true", help="skip the side workloads (other configurations, fairness sweep, probes)")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="only run the plain copy kernel over a 64 MiB buffer five times (reference point for memory-traffic counters)")
    ap.add_argument("--zoo-ops", nargs="?", const="all", default=None, metavar="MODELS",
                    help="only this: per operator family of every zoo model (or of the comma-separated ones), launches, time and rates "
                         "of one forward pass, one launch at a time")
    ap.add_argument("--overlap-probe", action="store_true",
                    help="only: whether vector-ALU instructions hide behind matrix instructions on this device (a table on stderr)")
    ap.add_argument("--queue-probe", action="store_true",
                    help="only: how many kernels run side by side and what sharing a launch gains (paella_queue_concurrency_probe), as a table on stderr")
    ap.add_argument("--roofline-only", default=None, metavar="MODEL",
                    help="only the isolated per-launch timing of one forward pass of MODEL (the leg roofline.achieved comes from)")
    ap.add_argument("--full-device", default=None, metavar="MODEL",
                    help="only: the conv kernel with the device full (every conv layer of MODEL over 16 stacked inputs, one launch at a time); "
                         "under counter collection one untimed launch per layer")
    ap.add_argument("--fd-kw", type=int, default=0, help="with --full-device: waves per workgroup of every tap-major layer (default: the layer's own)")
    ap.add_argument("--fd-depth", type=int, default=0, help="with --full-device: chunks of operands in flight per wave (3, 4, 6, 8, 12; default 2)")
    ap.add_argument("--fd-only", default=None, help="with --full-device: comma-separated substrings of the layers to run, e.g. '17x17 768->192'")
    ap.add_argument("--fd-images", type=int, default=16)
    ap.add_argument("--fd-transform", action="store_true",
                    help="with --full-device: a per-channel scale-shift applied to the input of every layer that can take one (conv_mfma_pre_kernel)")
    ap.add_argument("--fd-one-tile", action="store_true", help="with --full-device: workgroups of one 32 x 32 tile throughout")
    ap.add_argument("--fd-burst", type=int, default=8, help="with --full-device: launches enqueued back to back per sample; the last one is timed")
    ap.add_argument("--counter-pass", default=None, metavar="MODEL",
                    help="only this: three forward passes of MODEL, one launch at a time with a synchronize after each (the leg to run "
                         "under `rocprofv3 --pmc`: nothing else is in flight and at most one dispatch is ever queued)")
    args = ap.parse_args()
    if args.gpus != 1:
        log("bench.py: this build serves from ONE GPU (one server process per GPU, no cross-GPU exchange); run with --gpus 1")
        sys.exit(2)

    from paella_amd import _abi, models, serve
    hip = _abi.hip()
    _abi.ops()
    if args.copy_calibration:
        import torch
        n = 16 << 20  # floats: 64 MiB read + 64 MiB written per launch
        x = torch.ones(n, dtype=torch.float32, device="cuda:0")
        y = torch.empty_like(x)
        torch.cuda.synchronize()
        for _ in range(5):
            _abi.check(_abi.ops().paella_copy_launch(ctypes.c_void_p(x.data_ptr()), ctypes.c_void_p(y.data_ptr()), n, None, 0, None), "copy")
            torch.cuda.synchronize()
        print(json.dumps({"copy_calibration": {"launches": 5, "kib_read_per_launch": n * 4 / 1024, "kib_written_per_launch": n * 4 / 1024}}), flush=True)
        return
    if args.full_device:
        fd = full_device_pass(models, hip, args.full_device, images=args.fd_images, timed=not under_counter_collection(), kw=args.fd_kw, depth=args.fd_depth,
                              only=args.fd_only.split(",") if args.fd_only else None, burst=args.fd_burst, transform=args.fd_transform,
                              one_tile=args.fd_one_tile)
        for r in fd["layers"]:
            log("[bench] %-26s x%d  %5d workgroups x %d waves  %8.1f MFLOP  %s%s" % (r["layer"], r["count"], r["workgroups"], r["waves_per_workgroup"], r["flops"] / 1e6,
                "%7.2f us  %6.1f TFLOP/s" % (r["us"], r["flops"] / r["us"] / 1e6) if r["us"] else "", "  (input transformed)" if r["input_transformed"] else ""))
        if fd.get("achieved"):
            log("[bench] %s, layers weighted by count%s: %.1f TFLOP/s = %.1f %% of the fp32 MFMA peak" %
                (args.full_device, ", input transformed where the layer can" if args.fd_transform else "", fd["achieved"], 100 * fd["frac"]))
        print(json.dumps({"full_device": fd}), flush=True)
        return
    if args.counter_pass:
        ex = models.Exec(args.counter_pass, seed=1)
        stream = ctypes.c_void_p()
        hip.llis_hip_stream_create(ctypes.byref(stream))
        work = [ex.stage_work(i) for i in range(ex.num_stages)]
        for _ in range(3):
            for i in range(ex.num_stages):
                ex.launch_stage(i, stream)
                hip.llis_hip_stream_synchronize(stream)
        hip.llis_hip_stream_destroy(stream)
        ex.close()
        print(json.dumps({"counter_pass": {"model": args.counter_pass, "passes": 3,
                                           "stages": [{"op": w[0], "flops": w[1], "bytes": w[2]} for w in work]}}), flush=True)
        return
    if under_counter_collection():
        # A counter pass over `--zoo-ops arcfaceresnet100,densenet121` ended in a host-side segmentation fault inside the
        # profiler's packet interception (tens of thousands of dispatches queued without a synchronize between them);
        # the cause was not established, so the long legs refuse to run under counter collection.
        log("bench.py: counter collection is on (ROCPROF_COUNTERS is set): only --counter-pass MODEL and --copy-calibration run under it")
        sys.exit(2)
    if args.zoo_ops:
        # Isolated launches, so every figure contains the 4 us an empty kernel shows by these time stamps: operators
        # that read 4.0 us are at that floor, whatever their kernels do.
        wanted = models.names() if args.zoo_ops == "all" else args.zoo_ops.split(",")
        table = {}
        for m in wanted:
            r = conv_roofline(models, hip, m, 20)
            log("[bench] %-17s %3d launches, forward pass %7.1f us, back to back %6.0f passes/s" % (m, len(r["per_stage_us"]), r["forward_us"], r["direct_rps"]))
            table[m] = {"launches": len(r["per_stage_us"]), "forward_us": r["forward_us"], "back_to_back_passes_per_s": r["direct_rps"], "by_op": {}}
            for op, d in sorted(r["by_op"].items(), key=lambda kv: -kv[1]["us"]):
                row = {"launches": d["launches"], "us": d["us"], "us_per_launch": d["us"] / d["launches"], "tflops": d["flops"] / d["us"] / 1e6,
                       "gbytes_per_s": d["bytes"] / d["us"] / 1e3, "frac_of_fp32_mfma_peak": d["flops"] / d["us"] / 1e6 / FP32_MFMA_PEAK_TFLOPS,
                       "frac_of_hbm_peak": d["bytes"] / d["us"] / 1e3 / 8000.0}
                table[m]["by_op"][op] = row
                log("[bench]     %-8s %3d launches %8.1f us (%5.2f each)  %6.2f TFLOP/s (%4.1f%% of fp32 MFMA)  %7.1f GB/s (%4.1f%% of HBM)" %
                    (op, row["launches"], row["us"], row["us_per_launch"], row["tflops"], 100 * row["frac_of_fp32_mfma_peak"],
                     row["gbytes_per_s"], 100 * row["frac_of_hbm_peak"]))
        print(json.dumps({"zoo_ops": table}), flush=True)
        return
    if args.overlap_probe:
        lib = _abi.probes()
        out = {}
        log("[bench] four matrix instructions + N multiply-adds per iteration, eight waves per SIMD, register-resident (paella_mfma_valu_overlap_probe)")
        log("[bench] %4s %12s %14s %10s" % ("N", "both, us", "vector alone", "TFLOP/s"))
        for n in (0, 8, 16, 32, 64, 128):
            both, alone, tf = ctypes.c_double(), ctypes.c_double(), ctypes.c_double()
            _abi.check(lib.paella_mfma_valu_overlap_probe(n, ctypes.byref(both), ctypes.byref(alone), ctypes.byref(tf)), "paella_mfma_valu_overlap_probe")
            out[n] = {"us_both": both.value, "us_valu_alone": alone.value, "tflops": tf.value}
            log("[bench] %4d %12.1f %14.1f %10.1f" % (n, both.value, alone.value, tf.value))
        print(json.dumps({"mfma_valu_overlap": out}))
        return
    if args.queue_probe:
        from paella_amd._abi import ConvDesc
        lib = _abi.ops()
        shapes = [("Inception-v3 8x8 1280->320 1x1", 1280, 8, 320, 1, 0), ("Inception-v3 17x17 768->192 1x1", 768, 17, 192, 1, 0),
                  ("Inception-v3 35x35 288->64 1x1", 288, 35, 64, 1, 0), ("ResNet-18 14x14 256->256 3x3", 256, 14, 256, 3, 1),
                  ("ResNet-18 56x56 64->64 3x3", 64, 56, 64, 3, 1), ("ResNet-18 7x7 512->512 3x3", 512, 7, 512, 3, 1)]
        cases = [("1 queue, no barrier bit", 1, 1, 0), ("1 queue, barrier bit", 1, 1, 1), ("2 queues", 1, 2, 1), ("4 queues", 1, 4, 1), ("8 queues", 1, 8, 1),
                 ("4 queues, 2 per launch", 2, 4, 1), ("4 queues, 4 per launch", 4, 4, 1)]
        out = {}
        log("[bench] 16 independent instances of one conv layer, microseconds per conv (200 rounds):")
        log("[bench] %-34s " % "layer" + " ".join("%24s" % c[0] for c in cases))
        for name, c, hw, k, r, pad in shapes:
            d = ConvDesc(c, hw, hw, k, r, r, 1, 1, pad, pad, 1, 1, 1, 1, 0.0, 0.0)
            row = []
            for label, per, nq, ordered in cases:
                us = ctypes.c_double()
                _abi.check(_abi.probes().paella_queue_concurrency_probe(ctypes.byref(d), 16, per, nq, ordered, 200, ctypes.byref(us)), "paella_queue_concurrency_probe")
                row.append(us.value)
            out[name] = dict(zip([c[0] for c in cases], row))
            log("[bench] %-34s " % name + " ".join("%24.2f" % v for v in row))
        print(json.dumps({"queue_probe_us_per_conv": out}))
        return
    if args.roofline_only:
        rl = conv_roofline(models, hip, args.roofline_only, reps=50)
        out = {"roofline": roofline_of(rl, args.roofline_only), "per_stage_us": rl["per_stage_us"], "work": rl["work"],
               "forward_us": rl["forward_us"], "back_to_back_passes_per_s": rl["direct_rps"]}
        print(json.dumps(out), flush=True)
        return

    serve.lib()
    os.environ.setdefault("LLIS_MODEL_SEED", "1")
    os.environ["PAELLA_INPUT_RESIDENT"] = "0"   # every request's input crosses PCIe
    if args.no_verify:
        Arm.verify = 0
    ek, streams = args.extra_kernels, args.num_streams
    tenants = MIX
    cap = sum(t[4] for t in tenants)

    # The isolated per-launch timing goes first: after a minute of serving arms the same launches measure about 4 %
    # longer (the part has been under sustained load by then).
    rl = conv_roofline(models, hip, "inception_v3", reps=30)
    rl18 = conv_roofline(models, hip, "resnet18", reps=50)
    roofline = roofline_of(rl, "inception_v3")
    log("[bench] conv launches alone: Inception-v3 %.2f TFLOP/s (%.1f%% of fp32 MFMA peak, %.2f us per launch); ResNet-18 %.2f TFLOP/s (%.2f us per launch)" %
        (roofline["achieved"], 100 * roofline["frac"], roofline["us_per_launch_avg"], roofline_of(rl18, "resnet18")["achieved"], rl18["conv_us"] / rl18["conv_launches"]))

    # ---- the unit of each tenant's SLO: its latency alone, one request outstanding
    alone = {"small_cnn": alone_latency(serve, "tvm_mnist", 28 * 28, 10, 4000, ek, streams),
             "inception_v3": alone_latency(serve, "tvm_inception_v3", 3 * 299 * 299, 1000, 400, ek, streams)}
    slo_us = {k: SLO_FACTOR * v["p50_us"] for k, v in alone.items()}
    log("[bench] alone: small CNN p50 %.1f us, Inception-v3 p50 %.1f us -> p99 SLO %.0f us and %.0f us" %
        (alone["small_cnn"]["p50_us"], alone["inception_v3"]["p50_us"], slo_us["small_cnn"], slo_us["inception_v3"]))

    # ---- headline: full3, kernels on direct dispatch
    searches = {}
    with Arm(serve, "full3", "full3", "direct", streams, tenants, ek, unfair=args.unfair) as arm:
        rate, sat, pts = search_rate(arm, tenants, slo_us)
        searches["full3"] = {"saturation_rps": sat, "points": pts, "rate_at_slo_rps": rate}
        if rate is None:
            rate = 0.05 * sat
        n_timed, n_warm = args.steps * STEP_REQUESTS, args.warmup * STEP_REQUESTS
        final, attempts = None, []
        for attempt in range(10):
            r = arm.run(1e6 / rate, n_timed, n_warm)
            p = point_of(r, tenants, rate)
            p["meets_slo"] = meets(p, tenants, slo_us)
            attempts.append(p)
            final = (r, p)
            log("[bench] timed run at %.0f req/s offered: %.0f served over %.2f s, p99 %s -> %s" %
                (rate, r["throughput_rps"], r["elapsed_us"] / 1e6, " / ".join("%.0f" % p[t[0] + "_p99_us"] for t in tenants),
                 "SLO met" if p["meets_slo"] else "SLO missed"))
            if p["meets_slo"]:
                break
            rate *= 0.98  # the longer run saw a tail the search point did not: back off and measure again
        main_run, main_point = final
    # a rate at which a single answer was wrong is not a rate at which the SLO was met
    value = main_run["throughput_rps"] if main_point["meets_slo"] and not main_run.get("mismatches") else None

    # ---- the same search for plain multi-stream serving, served (fifo, job by job on HIP streams) and without a server
    arms_at_equal_load, equal_rate = {}, None
    if not args.no_arms:
        # policy and launch path apart: every scheduler on direct dispatch AND on HIP launches ("plain per-model stream serving"
        # is fifo: a whole request on one stream -- HIP streams by default, ordered direct-dispatch queues as fifo_direct_dispatch)
        for label, sched, dispatch, nstreams in [("fifo2_direct_dispatch", "fifo2", "direct", streams), ("fifo_direct_dispatch", "fifo", "direct", cap),
                                                 ("full3_hip_launch", "full3", "hip", streams), ("fifo2_hip_launch", "fifo2", "hip", streams),
                                                 ("fifo_multi_stream", "fifo", "hip", cap), ("direct_multi_stream", "direct", "hip", cap)]:
            with Arm(serve, label, sched, dispatch, nstreams, tenants, ek) as arm:
                rate_b, sat_b, pts_b = search_rate(arm, tenants, slo_us)
                searches[label] = {"saturation_rps": sat_b, "points": pts_b, "rate_at_slo_rps": rate_b}
                log("[bench] %s: saturation %.0f req/s, highest rate meeting the SLO: %s" % (label, sat_b, "%.0f req/s" % rate_b if rate_b else "none of the rates tried"))
        # every arm at ONE offered load: 80 % of the headline rate
        equal_rate = 0.8 * (value or main_run["throughput_rps"])
        for label, sched, dispatch, nstreams in [("full3_direct_dispatch", "full3", "direct", streams), ("full3_hip_launch", "full3", "hip", streams),
                                                 ("fifo2_direct_dispatch", "fifo2", "direct", streams), ("fifo2_hip_launch", "fifo2", "hip", streams),
                                                 ("fifo_direct_dispatch", "fifo", "direct", cap),
                                                 ("fifo_multi_stream", "fifo", "hip", cap), ("fifo_single_stream", "fifo", "hip", 1),
                                                 ("direct_multi_stream", "direct", "hip", cap)]:
            with Arm(serve, label, sched, dispatch, nstreams, tenants, ek) as arm:
                p = point_of(arm.run(1e6 / equal_rate, SEARCH_REQUESTS, 512), tenants, equal_rate)
                p["meets_slo"] = meets(p, tenants, slo_us)
                arms_at_equal_load[label] = p
                log("[bench]   at %.0f req/s offered, %-22s served %8.0f, p50 %s us, p99 %s us" %
                    (equal_rate, label, p["achieved_rps"], " / ".join("%.0f" % p[t[0] + "_p50_us"] for t in tenants),
                     " / ".join("%.0f" % p[t[0] + "_p99_us"] for t in tenants)))

    # ---- side workloads: the other benchmark configurations
    side = {}
    if not args.no_side:
        import numpy as np

        def one_model(model, adapter):
            t = [(model, adapter, model, 1.0, 32)]
            res = {}
            for mode in ("0", "1"):
                os.environ["PAELLA_INPUT_RESIDENT"] = mode
                with Arm(serve, "full3", "full3", "direct", streams, t, ek) as arm:
                    # (with resident inputs a pooled server-side instance keeps the input of its first request whatever slot it
                    # serves later: a measurement mode whose outputs are not the requests' own, so nothing is compared there)
                    res["pcie_inclusive" if mode == "0" else "input_resident"] = arm.run(0.0, 4096, 512, verify=None if mode == "0" else 0)["throughput_rps"]
            os.environ["PAELLA_INPUT_RESIDENT"] = "0"
            return res

        # configuration 2: ResNet-18 alone -- saturation, and the top of its published sweep (2000 req/s Poisson)
        r18 = one_model("resnet18", "tvm_resnet18")
        t18 = [("resnet18", "tvm_resnet18", "resnet18", 1.0, 32)]
        with Arm(serve, "full3", "full3", "direct", streams, t18, ek) as arm:
            r18["poisson_2000_rps"] = point_of(arm.run(1e6 / 2000.0, 4096, 256), t18, 2000.0)
            r18["poisson_at_0.8_of_saturation"] = point_of(arm.run(1e6 / (0.8 * r18["pcie_inclusive"]), 8192, 512), t18, 0.8 * r18["pcie_inclusive"])
        with Arm(serve, "fifo_multi_stream", "fifo", "hip", 32, t18, ek) as arm:
            r18["fifo_multi_stream_saturation_rps"] = arm.run(0.0, 4096, 512)["throughput_rps"]
        side["resnet18_alone"] = r18
        log("[bench] ResNet-18 alone: %.0f req/s with the input copy, %.0f with inputs resident; fifo multi-stream %.0f; at 2000 req/s p99 %.0f us" %
            (r18["pcie_inclusive"], r18["input_resident"], r18["fifo_multi_stream_saturation_rps"], r18["poisson_2000_rps"]["p99_us"]))

        # configurations 4 and 5: full3 against multi-stream fifo at 80 % of the lower saturation rate
        def mix_side(key, ten):
            sat = {}
            for label, sched, dispatch, ns in [("full3", "full3", "direct", streams), ("fifo_multi_stream", "fifo", "hip", sum(t[4] for t in ten))]:
                with Arm(serve, label, sched, dispatch, ns, ten, ek) as arm:
                    sat[label] = arm.run(0.0, 3072, 256)["throughput_rps"]
            rate = 0.8 * min(sat.values())
            res = {"saturation_rps": sat, "offered_rps": rate}
            for label, sched, dispatch, ns in [("full3", "full3", "direct", streams), ("fifo_multi_stream", "fifo", "hip", sum(t[4] for t in ten))]:
                with Arm(serve, label, sched, dispatch, ns, ten, ek) as arm:
                    res[label] = point_of(arm.run(1e6 / rate, 4096, 256), ten, rate)
            side[key] = res
            log("[bench] %s: saturation full3 %.0f / fifo %.0f req/s; at %.0f req/s p99 full3 %.0f us, fifo %.0f us" %
                (key, sat["full3"], sat["fifo_multi_stream"], rate, res["full3"]["p99_us"], res["fifo_multi_stream"]["p99_us"]))

        mix_side("mobilenetv2_resnet50_equal_rates", [("mobilenetv2", "tvm_mobilenet", "mobilenetv2", 0.5, 24), ("resnet50", "tvm_resnet50", "resnet50", 0.5, 24)])
        eight = [("densenet121", "densenet121"), ("googlenet", "googlenet"), ("squeezenet1_1", "squeezenet1_1"), ("resnet34", "resnet34"),
                 ("ultraface320", "ultraface320"), ("arcfaceresnet100", "arcfaceresnet100"), ("mobilenet", "mobilenetv2"), ("mnist", "mnist")]
        mix_side("eight_models_uniform", [(z, "tvm_" + a, z, 0.125, 8) for a, z in eight])

        # configuration 1: one client, one request at a time, small CNN, 10 000 requests
        side["small_cnn_closed_loop"] = alone_latency(serve, "tvm_mnist", 28 * 28, 10, 10000, ek, streams)
        log("[bench] small CNN closed loop: mean %.1f us, p50 %.1f us, p99 %.1f us per request" %
            (side["small_cnn_closed_loop"]["mean_us"], side["small_cnn_closed_loop"]["p50_us"], side["small_cnn_closed_loop"]["p99_us"]))

        # the reference client's default arrival process is log-normal (reference app/client.cpp:133-134): the headline
        # mix at half its SLO rate, in bursts (sigma 1.5)
        with Arm(serve, "full3", "full3", "direct", streams, tenants, ek) as arm:
            half = 0.5 * (value or main_run["throughput_rps"])
            jobs = [(serve.job_path(t[1]), t[3], t[4]) for t in tenants]
            r = serve.client_run(arm.srv.name, jobs, 1e6 / half, cap, 8192, warmup_jobs=512, dist="ln", ln_sigma=1.5, pin_threads=True)
            side["lognormal_arrivals_sigma_1.5"] = point_of(r, tenants, half)

        # The request ring's own latency (client -> server), the reference's PRINT_LAUNCH_JOB_IPC_LATENCY probe (reference
        # src/server/server.cpp:121-141): LAUNCH_JOB carries its send time, the server averages now - sent; the headline mix at half
        # its SLO rate, the first 1000 requests left out.
        os.environ["LLIS_IPC_LATENCY_SKIP"] = "1000"
        os.environ["PAELLA_DISPATCH"] = "direct"
        with serve.Server("bench%d_ipc" % os.getpid(), "full3", num_streams=streams, cpu=4, extra_kernels=ek, print_ipc_latency=True) as srv:
            half = 0.5 * (value or main_run["throughput_rps"])
            serve.client_run(srv.name, [(serve.job_path(t[1]), t[3], t[4]) for t in tenants], 1e6 / half, cap, 8192, warmup_jobs=512, pin_threads=True)
            mean_us, count = srv.ipc_latency()
        os.environ.pop("PAELLA_DISPATCH", None)
        side["launch_job_ipc_latency"] = {"mean_us": mean_us, "requests": count, "offered_rps": half}
        log("[bench] request ring: LAUNCH_JOB reaches the server %.2f us after the client sent it (mean of %d requests at %.0f req/s)" % (mean_us, count, half))

        # Deficit-threshold sweep (reference sosp23_artifact/gen_data_fig13.sh:37-60): ResNet-18 : Inception-v3 = 0.952 : 0.048 at
        # saturation, latency of each model over its latency alone, Jain's index over those slowdowns.
        from paella_amd import fairness
        fjobs = [("resnet18", "tvm_resnet18", "resnet18", 0.952, 119), ("inception_v3", "tvm_inception_v3", "inception_v3", 0.048, 6)]
        alone_f = []
        for t in fjobs:
            with Arm(serve, "full3", "full3", "direct", streams, [(t[0], t[1], t[2], 1.0, t[4])], ek) as arm:
                alone_f.append(arm.run(0.0, max(200, int(2000 * t[3])), 100)["all"]["mean"])
        sweep = {"workload": "ResNet-18 : Inception-v3 = 0.952 : 0.048, 119 + 6 outstanding, 2000 requests at saturation",
                 "alone_mean_latency_us": alone_f, "points": []}
        for f in (1.0, 100.0, 100000.0):
            os.environ["PAELLA_DISPATCH"] = "direct"
            name = "bench%d_fair_%d" % (os.getpid(), int(time.time() * 1000) % 100000)
            with serve.Server(name, "full3", num_streams=streams, cpu=4, extra_kernels=ek, unfair=f) as srv:
                r = serve.client_run(srv.name, [(serve.job_path(t[1]), t[3], t[4]) for t in fjobs], 0.0, 125, 2000, warmup_jobs=200, pin_threads=True)
            slow = [r["per_type"][i]["mean"] / alone_f[i] for i in range(2)]
            sweep["points"].append({"unfair": f, "requests_per_s": r["throughput_rps"], "slowdown": slow, "jain_index": float(fairness.jain_index(slow))})
            log("[bench]   unfair %-9g %.0f req/s, slowdown ResNet-18 %.2f, Inception-v3 %.2f, Jain index %.3f" %
                (f, r["throughput_rps"], slow[0], slow[1], sweep["points"][-1]["jain_index"]))
        os.environ.pop("PAELLA_DISPATCH", None)
        side["fairness_sweep"] = sweep

        # What the scheduling policy is worth once the launch path is equal: the reference's two-model workload (reference
        # sosp23_artifact/gen_data_fig12_paella.sh:62-84: ResNet-18 0.952 / 119 instances, Inception-v3 0.048 / 6, 125 outstanding at
        # most, log-normal arrivals) through full3, fifo2 and fifo, all three on direct dispatch, plus fifo on HIP streams; the
        # reference sweeps the mean inter-arrival time over 2222 ... 40000 us on its GPU, here the offered rate is 0.5, 0.8 and 0.95
        # of what full3 serves at saturation, sigma 1.5.
        pol = {"workload": "ResNet-18 : Inception-v3 = 0.952 : 0.048, 119 + 6 instances, log-normal arrivals (sigma 1.5), 8192 requests per point",
               "arms": {}}
        with Arm(serve, "full3", "full3", "direct", streams, fjobs, ek) as arm:
            pol["saturation_rps_full3"] = arm.run(0.0, 6144, 512)["throughput_rps"]
        for label, sched, dispatch, ns in [("full3_direct_dispatch", "full3", "direct", streams), ("fifo2_direct_dispatch", "fifo2", "direct", streams),
                                           ("fifo_direct_dispatch", "fifo", "direct", 125), ("fifo_multi_stream", "fifo", "hip", 125)]:
            pts = []
            with Arm(serve, label, sched, dispatch, ns, fjobs, ek) as arm:
                jobs = [(serve.job_path(t[1]), t[3], t[4]) for t in fjobs]
                for frac in (0.5, 0.8, 0.95):
                    rate = frac * pol["saturation_rps_full3"]
                    r = serve.client_run(arm.srv.name, jobs, 1e6 / rate, 125, 8192, warmup_jobs=512, dist="ln", ln_sigma=1.5, pin_threads=True, verify=Arm.verify)
                    if Arm.verify:
                        Arm.verified += r["verified_requests"]
                        Arm.mismatches += r["mismatches"]
                    p = point_of(r, fjobs, rate)
                    p["fraction_of_full3_saturation"] = frac
                    pts.append(p)
                    log("[bench]   policy %-22s at %.2f of saturation (%6.0f req/s): served %6.0f, p99 ResNet-18 %7.0f us, Inception-v3 %7.0f us" %
                        (label, frac, rate, p["achieved_rps"], p["resnet18_p99_us"], p["inception_v3_p99_us"]))
            pol["arms"][label] = pts
        side["policy_reference_two_model_workload"] = pol

    # ---- kernel-level figures
    lib = _abi.ops()
    fd = full_device_pass(models, hip, "inception_v3")
    roofline["full_device"] = {k: fd[k] for k in ("achieved", "frac", "unit", "how")}
    log("[bench] conv kernel with the device full (Inception-v3's layers over 16 stacked inputs): %.1f TFLOP/s = %.1f%% of peak" % (fd["achieved"], 100 * fd["frac"]))
    if not args.no_side:
        try:
            mq = multi_queue_rate(models, "inception_v3", reps=60)
            roofline["under_load"] = {"forward_passes_per_s": mq, "conv_tflops": mq * rl["conv_flops"] / 1e12,
                                      "frac": mq * rl["conv_flops"] / 1e12 / FP32_MFMA_PEAK_TFLOPS,
                                      "how": "4 Inception-v3 forward passes in flight on 4 ordered direct-dispatch queues, no hooks, no scheduler"}
            # closed loop at two depths: 16 requests in flight is what the headline mix keeps (more of the large model in flight costs
            # the small one its p99), 32 is where the rate of the model alone stops growing (24: +6 %, 32: +8 %, 48: +7 % over 16)
            by_depth = {}
            for depth in (16, 32):
                with serve.Server("bench_inc%d_%d" % (depth, os.getpid()), "full3", num_streams=streams, cpu=4, extra_kernels=ek) as srv:
                    r = serve.client_run(srv.name, [(serve.job_path("tvm_inception_v3"), 1.0, depth)], 0.0, depth, 4000, warmup_jobs=400, pin_threads=True,
                                         verify=Arm.verify)
                if Arm.verify:
                    Arm.verified += r["verified_requests"]
                    Arm.mismatches += r["mismatches"]
                by_depth[depth] = r["throughput_rps"]
            best = max(by_depth, key=by_depth.get)
            served = by_depth[best]
            roofline["served"] = {"forward_passes_per_s": served, "conv_tflops": served * rl["conv_flops"] / 1e12,
                                  "frac": served * rl["conv_flops"] / 1e12 / FP32_MFMA_PEAK_TFLOPS,
                                  "requests_outstanding": best,
                                  "requests_per_s_by_requests_outstanding": {str(k): v for k, v in by_depth.items()},
                                  "frac_at_16_outstanding": by_depth[16] * rl["conv_flops"] / 1e12 / FP32_MFMA_PEAK_TFLOPS,
                                  "how": "Inception-v3 alone through full3 at saturation (closed loop with 16 and with 32 requests outstanding, the higher "
                                         "rate; input copy per request): conv launches of different requests packed into shared launches"}
            log("[bench] Inception-v3 alone through full3 at saturation: %.0f requests/s with 16 outstanding, %.0f with 32 = %.1f%% of peak over the conv work" %
                (by_depth[16], by_depth[32], 100 * roofline["served"]["frac"]))
            mq18 = multi_queue_rate(models, "resnet18")
            side["resnet18_four_passes_in_flight"] = {"forward_passes_per_s": mq18, "conv_tflops": mq18 * rl18["conv_flops"] / 1e12,
                                                      "frac_of_fp32_mfma_peak": mq18 * rl18["conv_flops"] / 1e12 / FP32_MFMA_PEAK_TFLOPS}
            log("[bench] 4 passes in flight (direct queues, no scheduler): Inception-v3 %.0f passes/s = %.1f%% of peak; ResNet-18 %.0f passes/s = %.1f%% of peak" %
                (mq, 100 * roofline["under_load"]["frac"], mq18, 100 * side["resnet18_four_passes_in_flight"]["frac_of_fp32_mfma_peak"]))
        except RuntimeError as ex:
            log("[bench]   direct-dispatch queues unavailable: %s" % ex)
    peak = ctypes.c_double()
    if _abi.probes().paella_mfma_peak_probe(ctypes.byref(peak)) == 0:
        roofline["peak_measured"] = peak.value  # register-resident fp32 MFMA loop on this box; `peak` stays the published figure
    floor = ctypes.c_double()
    if _abi.probes().paella_empty_kernel_probe(200, ctypes.byref(floor)) == 0 and floor.value > 0:
        # what the same time stamps report for a kernel that does nothing: every per-launch figure taken this way contains it
        roofline["empty_kernel_us"] = floor.value
    notify = {}
    ring = ctypes.c_void_p()
    if not args.no_side and lib.paella_ring_create(1024000, 1, ctypes.byref(ring)) == 0:
        import numpy as np
        us = ctypes.c_double()
        if lib.paella_ring_bench_drain(ring, 64, 6400, 50, 500, ctypes.byref(us)) == 0:
            notify["ring_drain_64_blocks_us_per_kernel"] = us.value
        flag, sync = ctypes.c_double(), ctypes.c_double()
        if lib.paella_ring_bench_pingpong(100, 2000, ctypes.byref(flag), ctypes.byref(sync), None) == 0:
            notify["launch_plus_flag_store_us"] = flag.value
            notify["launch_plus_stream_sync_us"] = sync.value
        n_echo = 5000
        rtt, one_way = np.zeros(n_echo), np.zeros(n_echo)
        if lib.paella_ring_bench_echo(ring, 500, n_echo, rtt.ctypes.data, one_way.ctypes.data) == 0:
            rtt.sort()
            notify["echo_round_trip_us"] = {"p50": float(rtt[n_echo // 2]), "p99": float(rtt[int(n_echo * 0.99)]),
                                            "what": "host flag store -> resident lane sees it -> ring message readable on the host"}
            log("[bench] notification: echo round trip p50 %.2f / p99 %.2f us" % (rtt[n_echo // 2], rtt[int(n_echo * 0.99)]))
            # One way, device -> host: the lane's clock sample just before its ring store, translated into the host's clock domain
            # by the runtime, against the host's sample when the message became readable.  The translation has been seen off by
            # microseconds either way, and no exchange over this same channel can calibrate it better than the round trip itself;
            # so the round trip is reported as the upper bound of the one-way latency, and the translated figure only when it is
            # physically possible (between zero and the round trip).
            ow = np.sort(one_way[one_way > -1e29])
            g2h = {"upper_bound_p50": float(rtt[n_echo // 2]), "upper_bound_p99": float(rtt[int(n_echo * 0.99)]),
                   "what": "device -> host one way is at most the echo round trip (which also holds the host -> device leg)"}
            if len(ow) >= n_echo // 2:
                p50, p99 = float(ow[len(ow) // 2]), float(ow[int(len(ow) * 0.99)])
                g2h["clock_translated"] = {"p50": p50, "p99": p99, "plausible": bool(0.0 < p50 < rtt[n_echo // 2])}
                log("[bench] notification: GPU -> host one way <= %.2f us (round trip); by translated device clock p50 %.2f / p99 %.2f us%s" %
                    (g2h["upper_bound_p50"], p50, p99, "" if g2h["clock_translated"]["plausible"] else " (not plausible: the clock translation is off)"))
            notify["gpu_to_host_us"] = g2h
        lib.paella_ring_destroy(ring)

    # ---- the CPU path beside it: the oracle's forward pass of both tenants on the host cores, combined at the mix's ratio
    cpu = cpu_torch = None
    if not args.no_cpu:
        big = cpu_baseline("inception_v3", args.cpu_seconds, max_passes=16)
        small = cpu_baseline("mnist", 1.0, max_passes=2000)
        per_request_s = 0.9 / small["value"] + 0.1 / big["value"]
        cpu = {"value": 1.0 / per_request_s, "unit": "requests/s", "cores": big["cores"], "kind": "port",
               "sample": "CPU oracle (float accumulate, OpenMP), same graphs and weights, batch 1: %s; %s; mix rate = 1/(0.9 t_small + 0.1 t_big)" %
                         (big["sample"], small["sample"]),
               "inception_v3_passes_per_s": big["value"], "small_cnn_passes_per_s": small["value"]}
        try:
            tb, ts = torch_cpu_baseline("inception_v3", min(args.cpu_seconds, 8.0)), torch_cpu_baseline("mnist", 1.0)
            if tb and ts:
                cpu_torch = {"value": 1.0 / (0.9 / ts["value"] + 0.1 / tb["value"]), "unit": "requests/s", "cores": tb["cores"], "kind": "port",
                             "sample": "torch CPU operators (oneDNN), same graphs and weights: %s; %s; combined the same way" % (tb["sample"], ts["sample"])}
        except Exception as ex:  # torch missing or an operator it lacks: the oracle figure stands alone
            log("[bench]   torch CPU baseline unavailable: %s" % ex)
        log("[bench] CPU: oracle %.2f req/s of the mix on %d threads%s" % (cpu["value"], cpu["cores"], "" if not cpu_torch else ", torch CPU operators %.1f req/s" % cpu_torch["value"]))

    elapsed_ms = main_run["elapsed_us"] / 1e3
    out = {
        "metric": METRIC,
        "value": value,
        "unit": "requests/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": elapsed_ms / args.steps,
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": "small CNN (1x1x28x28) : Inception-v3 (1x3x299x299) = 9 : 1, batch 1 fp32, seeded weights, open-loop Poisson arrivals, "
                               "H2D copy of every request's input and D2H of its output (PCIe-inclusive), full3 scheduler with %d streams, kernels on "
                               "direct dispatch; SLO: per-tenant p99 <= %.0f x the tenant's alone latency (small CNN <= %.0f us, Inception-v3 <= %.0f us); "
                               "a step = %d requests" % (streams, SLO_FACTOR, slo_us["small_cnn"], slo_us["inception_v3"], STEP_REQUESTS),
                   "slo_us": slo_us, "slo_factor": SLO_FACTOR, "alone_latency": alone, "requests_per_step": STEP_REQUESTS,
                   "timed_requests": args.steps * STEP_REQUESTS, "timed_seconds": elapsed_ms / 1e3, "pools": {t[0]: t[4] for t in tenants}},
        "offered_rps": main_point["offered_rps"],
        "latency_us": {k: main_point[k] for k in main_point if k.endswith("_us")},
        "slo_met": main_point["meets_slo"],
        "verified_requests": main_run.get("verified_requests"),  # of the timed run: warm-up and measured completions, each compared
        "mismatches": main_run.get("mismatches"),                # byte for byte with the idle server's answer for the same input
        "verified_requests_all_runs": Arm.verified, "mismatches_all_runs": Arm.mismatches,
        "timed_run_attempts": attempts,
        "rate_search": searches,
        "arms_at_equal_offered_load": {"offered_rps": equal_rate, "arms": arms_at_equal_load},
        "roofline": roofline,
        "roofline_resnet18": roofline_of(rl18, "resnet18"),
        "cpu_baseline": cpu,
        "cpu_baseline_torch": cpu_torch,
        "side_workloads": side,
        "per_op_us": {k: {"launches": v["launches"], "us": v["us"], "gflop": v["flops"] / 1e9, "mbytes": v["bytes"] / 1e6,
                          "tflops": v["flops"] / (v["us"] * 1e-6) / 1e12 if v["us"] else None,
                          "gbytes_per_s": v["bytes"] / (v["us"] * 1e-6) / 1e9 if v["us"] else None} for k, v in rl["by_op"].items()},
        "notify_us": notify,
    }
    emit(out)


def _short(x, digits=6):
    """Numbers to `digits` significant figures, recursively: the stdout line is read by a harness that keeps a few KB."""
    if isinstance(x, bool) or x is None:
        return x
    if isinstance(x, float):
        return float("%.*g" % (digits, x))
    if isinstance(x, dict):
        return {k: _short(v, digits) for k, v in x.items()}
    if isinstance(x, (list, tuple)):
        return [_short(v, digits) for v in x]
    return x


def headline(out):
    """The one stdout line: the contract's keys, the roofline and CPU-baseline objects and a handful of headline figures.  Everything
    else the run measured (the rate-search points, every arm at equal load, the side workloads, per-operator times) goes to
    the detail file and to stderr; this line stays under 4 KB whatever the run produced."""
    cfg, rf = out["config"], out.get("roofline") or {}
    line = {k: out[k] for k in ("metric", "value", "unit", "n_gpus", "steps", "warmup", "ms_per_step", "higher_is_better", "scaling", "vs_baseline", "dtype", "data")}
    line["config"] = {"workload": "small CNN : Inception-v3 (299x299) = 9 : 1, batch 1, fp32, open-loop Poisson, per-request H2D/D2H, full3 on direct dispatch",
                      "slo_us": cfg.get("slo_us"), "slo_factor": cfg.get("slo_factor"), "timed_requests": cfg.get("timed_requests"),
                      "timed_seconds": cfg.get("timed_seconds"), "pools": cfg.get("pools")}
    for k in ("offered_rps", "slo_met", "latency_us", "verified_requests", "mismatches"):
        if k in out:
            line[k] = out[k]
    r = {k: rf.get(k) for k in ("bound", "achieved", "peak", "unit", "frac", "traffic") if k in rf}
    r["kernel"] = "conv_mfma_kernel, conv_small_kernel, conv_tall_kernel (+ grouped forms), Inception-v3's conv launches one at a time"
    for k in ("flops_per_launch_avg", "us_per_launch_avg", "algorithmic_bytes_per_launch_avg", "peak_measured", "empty_kernel_us"):
        if k in rf:
            r[k] = rf[k]
    for k in ("served", "under_load", "full_device"):
        if isinstance(rf.get(k), dict):
            r[k] = {"frac": rf[k].get("frac"), "tflops": rf[k].get("conv_tflops", rf[k].get("achieved"))}
            if "requests_outstanding" in rf[k]:
                r[k]["requests_outstanding"] = rf[k]["requests_outstanding"]
                r[k]["frac_at_16_outstanding"] = rf[k].get("frac_at_16_outstanding")
    line["roofline"] = r
    for key in ("cpu_baseline", "cpu_baseline_torch"):
        c = out.get(key)
        if c:
            line[key] = {"value": c["value"], "unit": c["unit"], "cores": c["cores"], "kind": c["kind"], "sample": c["sample"][:200]}
        else:
            line[key] = None
    arms = {}
    for label, s in (out.get("rate_search") or {}).items():
        arms[label] = {"rate_at_slo_rps": s.get("rate_at_slo_rps"), "saturation_rps": s.get("saturation_rps")}
    line["arms"] = arms
    n = out.get("notify_us") or {}
    line["notify_us"] = {k: ({kk: vv for kk, vv in v.items() if kk in ("p50", "p99", "upper_bound_p50", "upper_bound_p99")} if isinstance(v, dict) else v)
                         for k, v in n.items()}
    pol = (out.get("side_workloads") or {}).get("policy_reference_two_model_workload")
    if pol:  # per arm at 0.8 of full3's saturation rate: served rate and per-model p99
        line["policy_at_0.8_sat"] = {a: {"rps": pts[1]["achieved_rps"], "p99_us": [pts[1]["resnet18_p99_us"], pts[1]["inception_v3_p99_us"]]}
                                     for a, pts in pol["arms"].items() if len(pts) > 1}
    line["detail"] = "gpurun_out/bench_detail.json"
    line = _short(line)
    text = json.dumps(line, separators=(",", ":"))
    # belt and braces: whatever a future key adds, the line that carries the metric is never the one that gets cut
    for drop in ("policy_at_0.8_sat", "arms", "notify_us", "cpu_baseline_torch", "latency_us"):
        if len(text) < 4000:
            break
        line.pop(drop, None)
        text = json.dumps(line, separators=(",", ":"))
    return text


def emit(out):
    detail_dir = os.path.join(ROOT, "gpurun_out")
    try:
        os.makedirs(detail_dir, exist_ok=True)
        with open(os.path.join(detail_dir, "bench_detail.json"), "w") as f:
            json.dump(out, f, indent=1)
    except OSError as ex:
        log("[bench] detail file not written: %s" % ex)
    log("[bench] detail: " + json.dumps(_short(out)))
    for ln in SUMMARY:
        print(ln, file=sys.stderr)
    sys.stderr.flush()
    print(headline(out), flush=True)


if __name__ == "__main__":
    main()
