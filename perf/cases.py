"""What a user of this framework has it do, as cases that can be timed.

Four kinds of work, each through the public entry points of `paella_amd`:

  serve    a server (full3, kernels on direct dispatch) under a saturating client: one or two tenants, a pool of request slots
           each, every input and output through the request ring -- what the framework is for.  One pass is one run of the
           client: it attaches, registers its job types, fills its pools and gets every request answered.
  single   the same server with one request outstanding: a lone client in a closed loop.
  request  a model without a server (`models.Exec`): inputs from host memory, the forward pass, outputs back in host memory;
           one request or several, one after the other on the default stream or each on a stream of its own.
  conv, dwconv, pool, dense
           one operator called on device tensors, as a job definition of the user's own calls it.

All of it is fp32 at batch 1, the only type and batch size that the framework takes.  Weights are seeded (the zoo's own
generator), inputs are drawn from N(0, 1) from the state's seed, or by the load generator from that seed.
"""
import os
import threading
import weakref

import numpy as np
import torch

from paella_amd import models, ops, serve

os.environ.setdefault("LLIS_MODEL_SEED", "1")

# Job definitions of the zoo models.
ADAPTERS = {"mnist": "tvm_mnist", "mobilenetv2": "tvm_mobilenet", "squeezenet1_1": "tvm_squeezenet1_1", "ultraface320": "tvm_ultraface320",
            "googlenet": "tvm_googlenet", "resnet18": "tvm_resnet18", "resnet34": "tvm_resnet34", "resnet50": "tvm_resnet50",
            "densenet121": "tvm_densenet121", "inception_v3": "tvm_inception_v3", "arcfaceresnet100": "tvm_arcfaceresnet100"}

# GFLOP of one forward pass, to bound what a drawn case costs.
GFLOP = {"mnist": 0.0016, "ultraface320": 0.156, "mobilenetv2": 0.602, "squeezenet1_1": 0.698, "googlenet": 3.165, "resnet18": 3.628,
         "densenet121": 5.668, "resnet34": 7.328, "resnet50": 8.178, "inception_v3": 11.426, "arcfaceresnet100": 24.179}

VARIANTS = 4  # distinct inputs per tenant in a serve case


def listed():
    return [
        # A lone client of the small CNN: the round trip of one request through rings, scheduler and kernels.
        {"name": "single_small_cnn", "kind": "single", "model": "mnist", "requests": 400},
        # The headline mix of the serving benchmark: small CNN : Inception-v3 = 9 : 1, pools of 96 and 16.
        {"name": "serve_small_cnn_inception", "kind": "serve", "model": "mnist", "pool": 96, "share": 0.9, "other": "inception_v3", "other_pool": 16,
         "requests": 8192},
        # Depthwise and bottleneck networks at equal rates, 24 slots each.
        {"name": "serve_mobilenet_resnet50", "kind": "serve", "model": "mobilenetv2", "pool": 24, "share": 0.5, "other": "resnet50", "other_pool": 24,
         "requests": 2048},
        # One network alone under load.
        {"name": "serve_resnet18", "kind": "serve", "model": "resnet18", "pool": 48, "share": 1.0, "other": "", "other_pool": 0, "requests": 4096},
        # One request without a server, smallest network to largest: latency and launches count.
        {"name": "request_small_cnn", "kind": "request", "model": "mnist", "requests": 1, "streams": 0},
        {"name": "request_mobilenetv2", "kind": "request", "model": "mobilenetv2", "requests": 1, "streams": 0},
        {"name": "request_densenet121", "kind": "request", "model": "densenet121", "requests": 1, "streams": 0},
        {"name": "request_inception_v3", "kind": "request", "model": "inception_v3", "requests": 1, "streams": 0},
        {"name": "request_arcface_r100", "kind": "request", "model": "arcfaceresnet100", "requests": 1, "streams": 0},
        # Eight requests in flight on eight streams, as a program with its own dispatch serves them.
        {"name": "requests_resnet50_8_streams", "kind": "request", "model": "resnet50", "requests": 8, "streams": 8},
        # A residual block's 3x3 convolution (ResNet-18, second stage).
        {"name": "conv3x3_128_28", "kind": "conv", "c": 128, "h": 28, "w": 28, "k": 128, "r": 3, "s": 3, "stride": 1, "residual": True},
        # A depthwise layer on a large feature map (MobileNetV2): memory-bound.
        {"name": "dwconv3x3_96_112", "kind": "dwconv", "c": 96, "h": 112, "w": 112, "r": 3, "stride": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["serve", "single", "request", "request", "request", "conv", "conv", "dwconv", "pool", "dense"])
    if kind == "single":
        model = rng.choice(list(ADAPTERS))
        return {"kind": kind, "model": model, "requests": min(_log_int(rng, 50, 1000), int(1000 / (0.5 + GFLOP[model])))}
    if kind == "serve":
        model, other = rng.choice(list(ADAPTERS)), rng.choice([""] + list(ADAPTERS))
        if other == model:
            other = ""
        share = rng.choice([0.5, 0.75, 0.9]) if other else 1.0
        per_request = share * GFLOP[model] + ((1 - share) * GFLOP[other] if other else 0)
        return {"kind": kind, "model": model, "pool": _log_int(rng, 8, 96), "share": share, "other": other, "other_pool": _log_int(rng, 8, 48) if other else 0,
                "requests": min(_log_int(rng, 1024, 8192), int(8000 / per_request))}
    if kind == "request":
        requests = _log_int(rng, 1, 16)
        return {"kind": kind, "model": rng.choice(list(ADAPTERS)), "requests": requests, "streams": rng.choice([0, 1, min(max(requests, 2), 8)]) if requests > 1 else 1}
    if kind == "conv":
        # The layers of the networks: large maps with few channels to small maps with many; whole channel blocks and ragged ones.
        h = _log_int(rng, 7, 149)
        c, k = (_log_int(rng, 16, min(1024, 24000 // h)) for _ in range(2))
        if rng.random() < 0.6:
            c, k = max(16, c // 16 * 16), max(16, k // 16 * 16)
        r, s = rng.choice([(1, 1), (1, 1), (3, 3), (3, 3), (5, 5), (1, 7), (7, 1)])
        while c * k * r * s > 2 ** 21:
            c, k = max(16, c // 2), max(16, k // 2)
        return {"kind": kind, "c": c, "h": h, "w": max(7, h + rng.choice([0, 0, -1, 3])), "k": k, "r": r, "s": s, "stride": rng.choice([1, 1, 2]),
                "residual": rng.random() < 0.3}
    if kind == "dwconv":
        h = _log_int(rng, 7, 150)
        return {"kind": kind, "c": _log_int(rng, 16, 960), "h": h, "w": max(7, h + rng.choice([0, 0, 1, 80])), "r": rng.choice([3, 3, 5]), "stride": rng.choice([1, 2])}
    if kind == "pool":
        h = _log_int(rng, 7, 150)
        return {"kind": kind, "c": _log_int(rng, 16, 512), "h": h, "w": max(7, h + rng.choice([0, 0, 1, 5])), "r": rng.choice([2, 3]), "stride": rng.choice([1, 2]),
                "average": rng.random() < 0.4}
    return {"kind": "dense", "c": _log_int(rng, 64, 25088), "k": _log_int(rng, 10, 1024)}


# ---------------------------------------------------------------- preparation

class _Held:
    """Something to be closed once nothing refers to it any more."""

    def __init__(self, thing, close):
        self.thing = thing
        weakref.finalize(self, close)


_server_lock = threading.Lock()
_server_ref = None
_servers = 0


def _server():
    """The process's server: started by the first state that needs one, stopped with the last."""
    global _server_ref, _servers
    with _server_lock:
        held = _server_ref() if _server_ref is not None else None
        if held is None:
            _servers += 1
            srv = serve.Server("perf%d_%d" % (os.getpid(), _servers), "full3", num_streams=128, extra_kernels=48, cpu=4)
            srv.__enter__()
            held = _Held(srv, srv.stop)
            _server_ref = weakref.ref(held)
        return held


def _floats(model):
    i, o = models.io_bytes(model)
    return i // 4, o // 4


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    if kind == "single":
        n_in, n_out = _floats(case["model"])
        return {"case": case, "server": _server(), "path": serve.job_path(ADAPTERS[case["model"]]), "x": rng.standard_normal(n_in, dtype=np.float32), "n_out": n_out}
    if kind == "serve":
        jobs = [(serve.job_path(ADAPTERS[case["model"]]), case["share"], case["pool"])]
        outs = [_floats(case["model"])[1]]
        if case["other"]:
            jobs.append((serve.job_path(ADAPTERS[case["other"]]), 1.0 - case["share"], case["other_pool"]))
            outs.append(_floats(case["other"])[1])
        return {"case": case, "server": _server(), "jobs": jobs, "outs": outs, "seed": seed % (1 << 30)}
    if kind == "request":
        execs = []
        for _ in range(case["requests"]):
            ex = models.Exec(case["model"])
            execs.append(_Held(ex, ex.close))
        n_in = _floats(case["model"])[0]
        return {"case": case, "execs": execs, "x": [rng.standard_normal(n_in, dtype=np.float32) for _ in execs],
                "streams": [torch.cuda.Stream() for _ in range(case["streams"])]}
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if kind in ("conv", "dwconv"):
        depthwise = kind == "dwconv"
        c, k = case["c"], case["c"] if depthwise else case["k"]
        r, s = case["r"], case["r"] if depthwise else case["s"]
        w = rng.standard_normal((k, 1 if depthwise else c, r, s), dtype=np.float32) * np.float32((2.0 / (r * s * (1 if depthwise else c))) ** 0.5)
        residual = bool(case.get("residual"))
        conv = ops.Conv2d(w, rng.standard_normal(k, dtype=np.float32) * np.float32(0.1), stride=case["stride"], pad=(r // 2, s // 2), groups=c if depthwise else 1,
                          act=ops.ACT_RELU6 if depthwise else ops.ACT_RELU, in_hw=(case["h"], case["w"]), has_residual=residual)
        p, q = conv.plan.P, conv.plan.Q
        return {"case": case, "conv": conv, "x": torch.randn(1, c, case["h"], case["w"], device="cuda", generator=gen),
                "residual": torch.randn(1, k, p, q, device="cuda", generator=gen) if residual else None}
    if kind == "pool":
        return {"case": case, "x": torch.randn(1, case["c"], case["h"], case["w"], device="cuda", generator=gen)}
    return {"case": case, "x": torch.randn(1, case["c"], device="cuda", generator=gen),
            "w": torch.randn(case["k"], case["c"], device="cuda", generator=gen) * (1.0 / case["c"]) ** 0.5, "bias": torch.randn(case["k"], device="cuda", generator=gen)}


# ---------------------------------------------------------------- one pass

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "single":
        out, _ = serve.client_single(state["server"].thing.name, state["path"], state["x"], state["n_out"], n=case["requests"])
        return out
    if kind == "serve":
        cap = sum(j[2] for j in state["jobs"])
        r = serve.client_run(state["server"].thing.name, state["jobs"], 0.0, cap, case["requests"], seed=state["seed"], pin_threads=True, verify=VARIANTS,
                             expected_bytes=4 * VARIANTS * sum(state["outs"]))
        at, outs = 0, []
        expected = r["expected"].view(np.float32)
        for n in state["outs"]:
            outs.append(expected[at:at + VARIANTS * n])
            at += VARIANTS * n
        return {"answers": outs, "verified": int(r["verified_requests"]), "mismatches": int(r["mismatches"])}
    if kind == "request":
        streams = state["streams"]
        for i, (ex, x) in enumerate(zip(state["execs"], state["x"])):
            ex.thing.set_input(x)
            ex.thing.forward(streams[i % len(streams)].cuda_stream if streams else None)
        for s in streams:
            s.synchronize()
        return [ex.thing.get_output() for ex in state["execs"]]
    if kind in ("conv", "dwconv"):
        return state["conv"](state["x"], residual=state["residual"])
    if kind == "pool":
        return ops.pool2d(state["x"], case["r"], case["stride"], pad=case["r"] // 2 if case["r"] == 3 else 0, is_avg=case["average"])
    return ops.dense(state["x"], state["w"], state["bias"], act=ops.ACT_RELU)


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    kind = case["kind"]
    if kind in ("single", "serve", "request"):
        tenants = [(case["model"], case.get("share", 1.0))]
        if case.get("other"):
            tenants.append((case["other"], 1.0 - case["share"]))
        total = {"bytes": 0.0, "flops": 0.0}
        for model, share in tenants:
            t, (i, o) = models.totals(model), models.io_bytes(model)
            total["bytes"] += 4 * t["params"] + share * case["requests"] * (i + o)
            total["flops"] += share * case["requests"] * t["flops"]
        return total
    if kind in ("conv", "dwconv"):
        depthwise = kind == "dwconv"
        c, k = case["c"], case["c"] if depthwise else case["k"]
        r, s = case["r"], case["r"] if depthwise else case["s"]
        p, q = ((case["h"] + 2 * (r // 2) - r) // case["stride"] + 1), ((case["w"] + 2 * (s // 2) - s) // case["stride"] + 1)
        per_channel = (1 if depthwise else c) * r * s
        return {"bytes": 4.0 * (c * case["h"] * case["w"] + k * per_channel + k + k * p * q * (2 if case.get("residual") else 1)), "flops": 2.0 * k * per_channel * p * q}
    if kind == "pool":
        pad = 1 if case["r"] == 3 else 0
        p, q = ((case[e] + 2 * pad - case["r"]) // case["stride"] + 1 for e in ("h", "w"))
        return {"bytes": 4.0 * case["c"] * (case["h"] * case["w"] + p * q), "flops": 1.0 * case["c"] * p * q * case["r"] ** 2}
    return {"bytes": 4.0 * (case["c"] * case["k"] + case["c"] + 2 * case["k"]), "flops": 2.0 * case["c"] * case["k"]}


def tolerance(case):
    # fp32 throughout.  A pool's maximum is one of its inputs; a single operator is one 32-bit sum per value; a network is tens of
    # such layers one behind the other, each of which passes its input's rounding on.
    if case["kind"] == "pool":
        return {"rel": 1e-6} if case["average"] else "exact"
    if case["kind"] in ("conv", "dwconv", "dense"):
        return {"rel": 1e-5}
    return {"rel": 2e-5}
