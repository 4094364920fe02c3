"""Workloads of the gfx950 execution backend, as a program runs them.

A case is one call (or one replay, one served burst, one stream) through the
package's public entry points: a kernel, a form, a number of threads and where
the columns live.  `listed` holds the fixed ones, `draw` gives more of the same
ranges.  Columns in device memory are torch tensors handed over as
`loom_amd.DeviceArray`s; 64-bit unsigned columns are int64 tensors of the same
bits.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import loom_amd
from loom_amd import abi, autotune, serve, workloads
from loom_amd.stream import Stream

# ---- the kernels and their forms -----------------------------------------------

# columns: bytes in and out per thread; ops: operations per thread on the inputs
# below (whole-configuration means of the lowered kernels: fib over n in [0, 90],
# Collatz over [1, 2^32), path-traced samples of the nine-sphere scene)
KERNELS = {
    "fib_u64": {"bytes": 16, "ops": 271.0},
    "fib_u32": {"bytes": 8, "ops": 141.0},
    "collatz_u64": {"bytes": 12, "ops": 1606.0},
    "threefry2x32_u32": {"bytes": 24, "ops": 187.0},
    "cubic_bisect_f32": {"bytes": 24, "ops": 300.0},
    "cubic_bisect_f64": {"bytes": 48, "ops": 700.0},
    "smallpt9_f32": {"bytes": 20, "ops": 3219.0},
}

# the predicated form under the reference's policy (what compact_function runs by
# default) and under sweeps; the regrouping form with in-wave refill (what
# hybrid_function runs by default), with queues, and within workgroups; "best" is
# the form the autotuner stored for the kernel
FORMS = ("best", "compact", "sweep", "hybrid", "queues", "groups8", "groups16")

TORCH = {np.dtype(np.uint32): torch.int32, np.dtype(np.int32): torch.int32,
         np.dtype(np.uint64): torch.int64, np.dtype(np.int64): torch.int64,
         np.dtype(np.float32): torch.float32, np.dtype(np.float64): torch.float64}

FRAME_SPP = 255  # samples of a pixel in the finished frame; a launch renders some of them


class Column(loom_amd.DeviceArray):
    """A torch tensor on the GPU as a device column."""

    def __init__(self, tensor, dtype):
        self.tensor = tensor
        self.dtype = np.dtype(dtype)
        self.n = tensor.numel()
        self.nbytes = self.n * self.dtype.itemsize
        self.ptr = tensor.data_ptr()

    def free(self):
        self.tensor = None


def _params(form, kernel):
    if form == "best":
        name, best = autotune.best_form(kernel)
        mode = abi.MODE_HYBRID if name == "hybrid" else abi.MODE_COMPACT
        return mode, {**best, "stats": False}
    mode = abi.MODE_COMPACT if form in ("compact", "sweep") else abi.MODE_HYBRID
    extra = {
        "compact": {},
        "sweep": {"reconv": abi.RECONV_SWEEP},
        "hybrid": {},
        "queues": {"regroup": abi.REGROUP_QUEUES},
        "groups8": {"regroup": abi.REGROUP_WORKGROUP, "regroup_waves": 8, "regroup_phase": 256},
        "groups16": {"regroup": abi.REGROUP_WORKGROUP, "regroup_waves": 16, "regroup_phase": 256},
    }[form]
    return mode, {**extra, "stats": False}


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)
    return g


def _samples(w, h, spp, seed):
    """Sample indices of one pass over a w x h frame: `spp` consecutive samples of
    every pixel, from a place of the pixel's FRAME_SPP that the seed chooses."""
    g = _generator(seed)
    first = torch.randint(0, FRAME_SPP - spp + 1, (w * h, 1), generator=g, device="cuda")
    sid = torch.arange(w * h, device="cuda").unsqueeze(1) * FRAME_SPP + first
    sid = sid + torch.arange(spp, device="cuda")
    return sid.to(torch.int32).reshape(-1)


def _inputs(case, seed):
    """Input columns as tensors on the GPU, with the values the kernel meets."""
    k, g = case["kernel"], _generator(seed)
    if k == "smallpt9_f32":
        w, h, spp = case["w"], case["h"], case["spp"]
        sid = _samples(w, h, spp, seed)
        return [sid, torch.full_like(sid, workloads.pt_job(w, h, FRAME_SPP))]
    n = case["n"]
    if k.startswith("fib"):
        # F(90) and F(47) are the last that fit 64 and 32 bits
        top, ty = (90, torch.int64) if k == "fib_u64" else (47, torch.int32)
        return [torch.randint(0, top + 1, (n,), generator=g, device="cuda", dtype=ty)]
    if k == "collatz_u64":
        return [torch.randint(1, 1 << 32, (n,), generator=g, device="cuda")]
    if k == "threefry2x32_u32":
        return [torch.randint(-(1 << 31), 1 << 31, (n,), generator=g, device="cuda").to(torch.int32)
                for _ in range(2)]
    # cubic coefficients as workloads.cubic_inputs draws them
    ty, bound = (torch.float32, 100.0) if k == "cubic_bisect_f32" else (torch.float64, 1e5)

    def uniform(lo, hi):
        u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
        return lo + (hi - lo) * u

    sign = torch.where(uniform(0, 1) < 0.5, -1.0, 1.0)
    return [(uniform(1.0, bound) * sign).to(ty)] + [uniform(-bound, bound).to(ty) for _ in range(3)]


def _threads(case):
    return case["w"] * case["h"] * case["spp"] if case["kernel"] == "smallpt9_f32" else case["n"]


def _columns(name, tensors):
    k = loom_amd.kernel(name)
    n = tensors[0].numel()
    outs = [torch.zeros(n, dtype=TORCH[np.dtype(dt)], device="cuda") for dt in k.outputs]
    return ([Column(t, dt) for t, dt in zip(tensors, k.inputs)],
            [Column(t, dt) for t, dt in zip(outs, k.outputs)], outs)


def _host(tensor, dtype):
    return np.ascontiguousarray(tensor.cpu().numpy()).view(dtype)


# ---- the cases -----------------------------------------------------------------

def listed():
    return [
        # one call on a few thousand host rows, as a first program makes it:
        # launches, waits and copies are all there is
        {"name": "call_host_4099", "kind": "host", "kernel": "fib_u64", "form": "hybrid", "n": 4099},
        # a short launch on resident columns (the fib configuration)
        {"name": "fib_1m", "kind": "run", "kernel": "fib_u64", "form": "best", "n": 1 << 20},
        # the Collatz configuration: long uneven threads, in the tuned form
        {"name": "collatz_16m", "kind": "run", "kernel": "collatz_u64", "form": "best", "n": 1 << 24},
        # the same kernel as hybrid_function runs it, at a size that fills no wave or
        # grid evenly
        {"name": "collatz_ragged", "kind": "run", "kernel": "collatz_u64", "form": "hybrid",
         "n": 1000003},
        # straight-line counter-based random numbers: the path is its columns
        {"name": "threefry_16m", "kind": "run", "kernel": "threefry2x32_u32", "form": "compact",
         "n": 1 << 24},
        # divergent double-precision root finding
        {"name": "cubic_f64_1m", "kind": "run", "kernel": "cubic_bisect_f64", "form": "hybrid",
         "n": 1000001},
        # the path tracer's whole frame (the headline), in the tuned form
        {"name": "frame_1024x768x64", "kind": "run", "kernel": "smallpt9_f32", "form": "best",
         "w": 1024, "h": 768, "spp": 64},
        # a preview pass: few threads, so the longest paths decide
        {"name": "frame_preview", "kind": "run", "kernel": "smallpt9_f32", "form": "hybrid",
         "w": 161, "h": 119, "spp": 4},
        # the predicated form as compact_function runs it (the reference's policy)
        {"name": "frame_compact", "kind": "run", "kernel": "smallpt9_f32", "form": "compact",
         "w": 320, "h": 240, "spp": 16},
        # uneven launches of three kernels captured into one graph and replayed
        {"name": "batch_16_jobs", "kind": "batch", "jobs": 16, "scale": 2},
        # a burst of launches from host columns through the serving loop
        {"name": "serve_burst", "kind": "serve", "requests": 20, "w": 192, "h": 160, "spp": 8,
         "n": 60001},
        # threads exchanged through resident slots, the reference's stream protocol
        {"name": "stream_collatz", "kind": "stream", "kernel": "collatz_u64", "n": 300007,
         "slots": 1 << 16},
    ]


def _between(rng, lo, hi):
    """A size spread over its logarithm, rarely a round number."""
    n = int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    return max(lo, min(hi, n))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "run", "run", "host", "batch", "serve", "stream"])
    if kind == "batch":
        return {"kind": "batch", "jobs": rng.randint(2, 16), "scale": rng.randint(2, 8)}
    if kind == "serve":
        return {"kind": "serve", "requests": rng.randint(4, 20), "w": rng.randint(32, 192),
                "h": rng.randint(32, 160), "spp": rng.randint(1, 8), "n": _between(rng, 512, 60001)}
    if kind == "stream":
        return {"kind": "stream", "kernel": rng.choice(["collatz_u64", "fib_u64", "cubic_bisect_f32"]),
                "n": _between(rng, 5000, 300007), "slots": 64 * _between(rng, 64, 1024)}
    if kind == "host":
        return {"kind": "host", "kernel": rng.choice([k for k in KERNELS if k != "smallpt9_f32"]),
                "form": rng.choice(["compact", "hybrid"]), "n": _between(rng, 64, 1 << 18)}
    kernel = rng.choice(["smallpt9_f32"] * 3 + list(KERNELS))
    form = rng.choice(FORMS)
    if kernel == "smallpt9_f32":
        # the slower forms on smaller frames, so that none takes longer than the whole frame
        top = 1024 if form in ("best", "hybrid") else 384
        return {"kind": "run", "kernel": kernel, "form": form, "w": _between(rng, 32, top),
                "h": _between(rng, 24, top * 3 // 4), "spp": _between(rng, 1, 64 if top > 384 else 16)}
    top = 1 << 24 if form in ("best", "hybrid", "sweep") else 1 << 21
    return {"kind": "run", "kernel": kernel, "form": form, "n": _between(rng, 64, top)}


# ---- what a program holds before the call ------------------------------------------

def _batch_specs(case):
    """The first jobs of the mixed benchmark batch, their sizes divided by `scale`."""
    specs = []
    for name, s in workloads.batch_jobs(case["jobs"], scale=case["scale"]):
        specs.append({"kernel": name, **{k: s[k] for k in ("w", "h", "spp", "n") if k in s}})
    return specs


def _serve_specs(case):
    """Frames (rows of one frame size), fib and Collatz launches, in turn."""
    specs = []
    for i in range(case["requests"]):
        if i % 2 == 0:
            rows = max(1, case["h"] * (1 + i % 5) // 5)
            specs.append(serve.RequestSpec("smallpt9_f32", case["w"] * rows * case["spp"], 0.0,
                                           case["w"], case["h"], FRAME_SPP))
        else:
            n = max(1, case["n"] * (1 + i % 7) // 7)
            specs.append(serve.RequestSpec("fib_u64" if i % 4 == 1 else "collatz_u64", n, 0.0,
                                           offset=(case["n"] - n) // 2))
    return specs


def prepare(case, seed):
    loom_amd.init(0)
    kind = case["kind"]
    if kind == "host":
        k = loom_amd.kernel(case["kernel"])
        ins = [_host(t, dt) for t, dt in zip(_inputs(case, seed), k.inputs)]
        f = (loom_amd.compact_function if case["form"] == "compact" else loom_amd.hybrid_function)(
            case["kernel"])
        return {"kind": kind, "f": f, "ins": ins}
    if kind == "run":
        ins, outs, tensors = _columns(case["kernel"], _inputs(case, seed))
        mode, params = _params(case["form"], case["kernel"])
        return {"kind": kind, "k": loom_amd.kernel(case["kernel"]), "mode": mode, "ins": ins,
                "outs": outs, "tensors": tensors, "params": loom_amd.make_params(mode=mode, **params)}
    if kind == "batch":
        b, tensors = loom_amd.Batch("pt_int_mix"), []
        for i, s in enumerate(_batch_specs(case)):
            ins, outs, t = _columns(s["kernel"], _inputs(s, seed + 7919 * (i + 1)))
            b.add(s["kernel"], ins, outs, 0, t[0].numel())
            tensors.append(t)
        params = loom_amd.make_params(mode=abi.MODE_HYBRID, stats=False,
                                      **autotune.best_params("batch:pt_int_mix"))
        torch.cuda.synchronize()
        return {"kind": kind, "graph": b.graph(params), "tensors": tensors}
    if kind == "serve":
        pools = serve.Pools()
        sid = _samples(case["w"], case["h"], case["spp"], seed)
        pools.sid = serve.Pinned(sid.numel(), np.uint32)
        pools.sid.array[:] = _host(sid, np.uint32)
        for name, k in (("fib", "fib_u64"), ("collatz", "collatz_u64")):
            pool = serve.Pinned(case["n"], np.uint64)
            pool.array[:] = _host(_inputs({"kernel": k, "n": case["n"]}, seed + 1)[0], np.uint64)
            setattr(pools, name, pool)
        specs = _serve_specs(case)
        outs = [[serve.Pinned(s.n, dt) for dt in loom_amd.kernel(s.kernel).outputs] for s in specs]
        return {"kind": kind, "specs": specs, "pools": pools, "pinned": outs,
                "outs": [[p.array for p in o] for o in outs],
                "server": serve.Server(hbm_budget=1 << 30)}
    k = loom_amd.kernel(case["kernel"])
    return {"kind": kind, "stream": Stream(case["kernel"], case["slots"], stats=False),
            "ins": [_host(t, dt) for t, dt in zip(_inputs(case, seed), k.inputs)]}


def _signed(columns):
    """Host columns with unsigned words as signed ones of the same bits."""
    return [c.view(c.dtype.str.replace("u", "i")) for c in columns]


def run(state):
    kind = state["kind"]
    if kind == "host":
        return _signed(state["f"](*state["ins"]))
    if kind == "run":
        loom_amd.run(state["k"], state["mode"], state["ins"], state["outs"], params=state["params"])
        return state["tensors"]
    if kind == "batch":
        state["graph"].launch()
        return state["tensors"]
    if kind == "serve":
        requests, _, outs = state["server"].run(state["specs"], state["pools"], realtime=False,
                                                outputs=state["outs"])
        if any(q.status for q in requests):
            raise RuntimeError("a request failed")
        # copies: the pinned columns are the state's own and go with it
        return [_signed([c.copy() for c in o]) for o in outs]
    return _signed(state["stream"].run_all(state["ins"]))


# ---- what a pass cannot do without ---------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("batch", "serve"):
        specs = (_batch_specs(case) if kind == "batch" else
                 [{"kernel": s.kernel, "n": s.n} for s in _serve_specs(case)])
        jobs = [(s["kernel"], s["n"]) for s in specs]
    else:
        jobs = [(case["kernel"], _threads(case))]
    return {"bytes": float(sum(KERNELS[k]["bytes"] * n for k, n in jobs)),
            "flops": float(sum(KERNELS[k]["ops"] * n for k, n in jobs))}


def tolerance(case):
    # the op contract fixes every bit: IEEE round-to-nearest without contraction,
    # whole numbers modulo their width
    return "exact"


# ---- the same in plain torch, in 64 bits ----------------------------------------------

def _fib(n, bits):
    table, a, b = [], 0, 1
    for i in range(91):
        # F(0) = 0 and F(1) = 1: what the kernel gives for n <= 1 is n
        table.append(a % (1 << bits))
        a, b = b, a + b
    table = [v - (1 << bits) if v >= 1 << (bits - 1) else v for v in table]
    return torch.tensor(table, device="cuda")[n.to(torch.int64)]


def _collatz(x):
    """Steps to 1 (starts below 2^32 stay below 2^63)."""
    x = x.clone()
    steps = torch.zeros_like(x)
    where = torch.arange(x.numel(), device="cuda")
    where, x = where[x > 1], x[x > 1]
    t = 0
    while x.numel():
        x = torch.where(x % 2 == 0, x // 2, 3 * x + 1)
        t += 1
        done = x == 1
        if t % 8 == 0 or bool(done.any()):
            steps[where[done]] = t
            where, x = where[~done], x[~done]
    return steps.to(torch.int32)


def _threefry(c0, c1):
    """Threefry-2x32 with 32 rounds, key (0xdead, 0xbeef), and the counter advanced."""
    m = 0xFFFFFFFF
    c0, c1 = c0.to(torch.int64) & m, c1.to(torch.int64) & m
    key = [0xdead, 0xbeef, 0x1bd11bda ^ 0xdead ^ 0xbeef]
    x0, x1 = (c0 + key[0]) & m, (c1 + key[1]) & m
    for r in range(32):
        left = (13, 15, 26, 6, 17, 29, 16, 24)[r % 8]
        x0 = (x0 + x1) & m
        x1 = (((x1 << left) & m) | (x1 >> (32 - left))) ^ x0
        if r % 4 == 3:
            s = r // 4 + 1
            x0 = (x0 + key[s % 3]) & m
            x1 = (x1 + key[(s + 1) % 3] + s) & m
    n0 = (c0 + 39916801) & m
    n1 = (c1 + (n0 < c0).to(torch.int64)) & m
    return [torch.where(v >= 1 << 31, v - (1 << 32), v).to(torch.int32) for v in (x0, x1, n0, n1)]


def _reference(kernel, ins):
    """Outputs of a kernel, None where 64 bits have no answer of their own: a path-
    traced sample and a bisection in 32 bits go where 32-bit values send them."""
    if kernel.startswith("fib"):
        bits = 64 if kernel == "fib_u64" else 32
        return [_fib(ins[0], bits).to(torch.int64 if bits == 64 else torch.int32)]
    if kernel == "collatz_u64":
        return [_collatz(ins[0])]
    if kernel == "threefry2x32_u32":
        return _threefry(*ins)
    if kernel == "cubic_bisect_f64":
        a, b, c, d = ins

        def at(x):
            return a * x * x * x + (b * x * x + (c * x + d))

        lo, hi = torch.full_like(a, -10.0), torch.full_like(a, 10.0)
        for _ in range(39):
            grow = (at(lo) < 0) == (at(hi) < 0)
            if not bool(grow.any()):
                break
            lo, hi = torch.where(grow, lo * 10, lo), torch.where(grow, hi * 10, hi)
        for _ in range(257):
            mid = lo + (hi - lo) * 0.5
            far = at(mid).abs() >= 0.1
            if not bool(far.any()):
                break
            left = (at(lo) < 0) != (at(mid) < 0)
            hi = torch.where(far & left, mid, hi)
            lo = torch.where(far & ~left, mid, lo)
        return [mid, None]
    return [None] * len(loom_amd.kernel(kernel).outputs)


def exact(case, seed):
    loom_amd.init(0)
    kind = case["kind"]
    if kind == "batch":
        return [_reference(s["kernel"], _inputs(s, seed + 7919 * (i + 1))
                           if s["kernel"] != "smallpt9_f32" else None)
                for i, s in enumerate(_batch_specs(case))]
    if kind == "serve":
        pool = {k: _inputs({"kernel": k, "n": case["n"]}, seed + 1)[0]
                for k in ("fib_u64", "collatz_u64")}
        return [_reference(s.kernel, None if s.kernel == "smallpt9_f32" else
                           [pool[s.kernel][s.offset:s.offset + s.n]]) for s in _serve_specs(case)]
    if case["kernel"] in ("smallpt9_f32", "cubic_bisect_f32"):
        return None
    return _reference(case["kernel"], _inputs(case, seed))
