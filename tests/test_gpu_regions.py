"""Runs that count no work sweep a kernel's regions (whole loops and branches
of small blocks) instead of its blocks.  Every output equals the oracle's bit
for bit over loops in loops, loops with several exits, jump tables and
straight lines, for sizes around a wave, refilled and not, and in the runs
that stay with blocks (a dispatch budget of their own)."""
import numpy as np
import pytest

import loom_amd
from loom_amd import abi, workloads
from loom_amd.stream import Stream
from tests import oracle_lib as O

pytestmark = pytest.mark.gpu


def words(n, seed):
    return np.random.default_rng(seed).integers(0, 1 << 32, n, dtype=np.uint32)


INPUTS = {
    "nested_u32": lambda n: [words(n, 1), words(n, 2)],
    "jump4_u32": lambda n: [words(n, 3) % np.uint32(6)],
    "factorial_u64": lambda n: [workloads.uniform_int(4, n, 0, 20)],
    "fib_u32": lambda n: [workloads.uniform_int(5, n, 0, 47).astype(np.uint32)],
    "collatz_u64": lambda n: [workloads.collatz_inputs(n, seed=6)],
    "cubic_bisect_f32": lambda n: workloads.cubic_inputs(n),
    "cubic_bisect_f64": lambda n: workloads.cubic_inputs(n, np.float64),
}
FORMS = {
    "compact": (abi.MODE_COMPACT, dict(reconv=abi.RECONV_SWEEP)),
    "refill": (abi.MODE_HYBRID, dict(live_threshold=48)),
    "refill late, one wave per CU": (abi.MODE_HYBRID, dict(live_threshold=1, waves_per_cu=1)),
    "queues": (abi.MODE_HYBRID, dict(regroup=abi.REGROUP_QUEUES)),
    "groups": (abi.MODE_HYBRID, dict(regroup=abi.REGROUP_WORKGROUP, regroup_phase=16)),
    "own budget": (abi.MODE_HYBRID, dict(max_steps=1 << 30)),
}


def bits(a):
    return a.view(np.uint32 if a.dtype.itemsize == 4 else np.uint64)


@pytest.mark.parametrize("name", list(INPUTS))
def test_regions_match_oracle(gpu, name):
    for n in (1, 63, 64, 65, 20011):
        ins = INPUTS[name](n)
        want, err = O.run(name, ins)
        assert err == 0
        for form, (mode, params) in FORMS.items():
            print(f"[gpu] regions {name} n={n} {form}", flush=True)
            r = loom_amd.run(name, mode, ins,
                             params=loom_amd.make_params(mode=mode, stats=False, **params))
            for g, w in zip(r.outputs, want):
                assert np.array_equal(bits(g), bits(w)), (name, n, form)


@pytest.mark.parametrize("name", ["nested_u32", "collatz_u64"])
def test_regions_in_streams_and_batches(gpu, name):
    ins = INPUTS[name](3001)
    want, _ = O.run(name, ins)
    for live in (0, 32):
        print(f"[gpu] region stream {name} live={live}", flush=True)
        s = Stream(name, 256, live_threshold=live, stats=False)
        for g, w in zip(s.run_all(ins), want):
            assert np.array_equal(bits(g), bits(w)), (name, live)
    if name != "collatz_u64":
        return
    k = loom_amd.kernel(name)
    b = loom_amd.Batch("int_mix")
    din = [loom_amd.DeviceArray.from_numpy(a) for a in ins]
    outs = [loom_amd.DeviceArray(3001, dt) for dt in k.outputs]
    b.add(k, din, outs)
    b.run(loom_amd.make_params(mode=abi.MODE_HYBRID, live_threshold=48, stats=False))
    assert np.array_equal(outs[0].numpy(), want[0])


def test_step_budget_still_trips(gpu):
    """A budget below the kernel's need is an error with and without
    statistics, and one above it is none."""
    ins = [np.full(64, 27, np.uint64)]
    for stats in (True, False):
        p = loom_amd.make_params(mode=abi.MODE_COMPACT, reconv=abi.RECONV_SWEEP, stats=stats,
                                 max_steps=50)
        with pytest.raises(abi.LoomError):
            loom_amd.run("collatz_u64", abi.MODE_COMPACT, ins, params=p)
        p.max_steps = 100000
        r = loom_amd.run("collatz_u64", abi.MODE_COMPACT, ins, params=p)
        assert (r.outputs[0] == 111).all()
