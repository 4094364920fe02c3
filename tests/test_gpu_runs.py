"""State that stays between runs on one context: input cursors that count on
from run to run, counters that are subtracted instead of cleared, error words
in host memory, pinned columns of small host calls.  Runs of different forms,
with and without statistics, failing ones among them, in one sequence: every
result and every count is that of the run alone."""
import ctypes as C

import numpy as np
import pytest

import loom_amd
from loom_amd import abi, workloads

pytestmark = pytest.mark.gpu

N = 16 * 256 * 64 + 333  # claims from ranges on a grid of one wave per CU
WORK = (abi.C_ACTIVE_OPS, abi.C_THREAD_STEPS)


def fib(n):
    a, b, t = 0, 1, []
    for _ in range(91):
        t.append(a)
        a, b = b, a + b
    return np.array(t, np.uint64)[n.astype(np.int64)]


def test_sequence_of_runs(gpu):
    x = workloads.fib_inputs(N, seed=17)
    want = fib(x)
    din = loom_amd.DeviceArray.from_numpy(x)
    steps = np.where(x <= 1, 1, x + 1).sum()
    forms = [("hybrid", dict(waves_per_cu=1)), ("hybrid", dict(regroup=abi.REGROUP_QUEUES)),
             ("hybrid", dict(regroup=abi.REGROUP_WORKGROUP, regroup_waves=8)),
             ("hybrid", dict(regroup=abi.REGROUP_WORKGROUP)), ("compact", dict(reconv=2)),
             ("batch", {}), ("fails", {})]
    rng = np.random.default_rng(18)
    with loom_amd.Context() as ctx:
        for i in range(60):
            form, params = forms[rng.integers(len(forms))]
            stats = bool(rng.integers(2))
            print(f"[gpu] run {i}: {form} {params} stats {stats}", flush=True)
            out = loom_amd.DeviceArray.full(N, 0xFFFFFFFFFFFFFFFF, np.uint64)
            if form == "fails":
                p = loom_amd.make_params(mode=abi.MODE_HYBRID, max_steps=3, stats=stats)
                with pytest.raises(abi.LoomError):
                    ctx.run("fib_u64", abi.MODE_HYBRID, [din], [out], params=p)
                continue
            if form == "batch":
                b, r = loom_amd.Batch("int_mix"), abi.RunStats()
                b.add("fib_u64", [din], [out])
                p = loom_amd.make_params(mode=abi.MODE_HYBRID, stats=stats)
                abi.check(abi.load().loom_ctx_batch_run(ctx.handle, b.set, b._table(), 1,
                                                        C.byref(p), C.byref(r)), "batch")
            else:
                m = abi.MODE_HYBRID if form == "hybrid" else abi.MODE_COMPACT
                r = ctx.run("fib_u64", m, [din], [out],
                            params=loom_amd.make_params(mode=m, stats=stats, **params))
            assert np.array_equal(out.numpy(), want), (i, form, params)
            assert r.errors == 0
            assert r.counters[abi.C_THREAD_STEPS] == (steps if stats else 0), (i, form, params)


def test_graph_between_runs(gpu):
    """Replays of a graph with statistics, other runs of its context between."""
    x = workloads.fib_inputs(5000, seed=19)
    din, out = loom_amd.DeviceArray.from_numpy(x), loom_amd.DeviceArray(5000, np.uint64)
    b = loom_amd.Batch("int_mix")
    b.add("fib_u64", [din], [out])
    g = b.graph(loom_amd.make_params(mode=abi.MODE_HYBRID))
    first = None
    for i in range(4):
        out.zero()
        r = g.launch()
        assert np.array_equal(out.numpy(), fib(x)), i
        counts = [r.counters[c] for c in WORK]
        first = first or counts
        assert counts == first, i
        alone = loom_amd.run("fib_u64", abi.MODE_COMPACT, [din], [out],
                             params=loom_amd.make_params(reconv=abi.RECONV_SWEEP))
        assert [alone.counters[c] for c in WORK] == first, i
        with pytest.raises(abi.LoomError):
            loom_amd.run("fib_u64", abi.MODE_HYBRID, [din], [out],
                         params=loom_amd.make_params(mode=abi.MODE_HYBRID, max_steps=2))


@pytest.mark.parametrize("total", [0, 1, 2])
def test_host_columns_around_the_pinned_size(gpu, total):
    """Two columns of 8 bytes at 2 MiB together, one element less and more."""
    n = (1 << 17) + total - 1
    x = workloads.fib_inputs(n, seed=20 + total)
    f = loom_amd.compact_function("fib_u64", reconv=abi.RECONV_SWEEP)
    assert np.array_equal(f(x)[0], fib(x))
    y = [np.random.default_rng(21).integers(0, 1 << 32, 300, dtype=np.uint32) for _ in range(2)]
    a = loom_amd.hybrid_function("int_mix_u32")(*y)
    dev = loom_amd.run("int_mix_u32", abi.MODE_COMPACT, [loom_amd.DeviceArray.from_numpy(c) for c in y])
    for g, d in zip(a, dev.outputs):
        assert np.array_equal(g, d.numpy())
    assert all(len(c) == 0 for c in f(np.zeros(0, np.uint64)))
