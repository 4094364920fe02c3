"""Refilling from a wave's pool of started threads (kernels with a long START,
sweep policy): outputs equal the oracle's bit for bit and every thread's work
is counted once, for inputs below a wave, a few rows past a pool, and many
pools per wave; refilled at any threshold, at the last lane and not at all; a
START that halts for some threads and goes several ways for others."""
import numpy as np
import pytest

import loom_amd
from loom_amd import abi, workloads
from tests import oracle_lib as O

pytestmark = pytest.mark.gpu


def started(n):
    rng = np.random.default_rng(n)
    return [rng.integers(0, 1 << 64, n, dtype=np.uint64) for _ in range(2)]


def frame(n):
    sid = np.arange(n, dtype=np.uint32) * np.uint32(7)
    return [sid, np.full(n, workloads.pt_job(61, 43, 255), np.uint32)]


def crowded(n):
    """For a kernel with too many words live after START for a pool."""
    return started(n)


INPUTS = {"started_u64": started, "smallpt9_f32": frame, "crowded_u64": crowded}
FORMS = [dict(live_threshold=48), dict(live_threshold=63), dict(live_threshold=0),
         dict(live_threshold=60, waves_per_cu=1), dict(refill=False),
         dict(live_threshold=32, reconv=abi.RECONV_TOPO)]
WORK = (abi.C_ACTIVE_OPS, abi.C_THREAD_STEPS, abi.C_ACTIVE_FLOPS)


def bits(a):
    return a.view(np.uint32) if a.dtype == np.float32 else a


@pytest.mark.parametrize("name", list(INPUTS))
def test_pool_matches_oracle(gpu, name):
    for n in (1, 63, 64, 65, 127, 129, 4 * 256 * 64 + 17):
        ins = INPUTS[name](n)
        want, err = O.run(name, ins)
        assert err == 0
        base = loom_amd.run(name, abi.MODE_COMPACT, ins,
                            params=loom_amd.make_params(reconv=abi.RECONV_SWEEP))
        for params in FORMS:
            for stats in (True, False):
                print(f"[gpu] pool {name} n={n} {params} stats {stats}", flush=True)
                r = loom_amd.run(name, abi.MODE_HYBRID, ins, params=loom_amd.make_params(
                    mode=abi.MODE_HYBRID, stats=stats, **params))
                for g, w in zip(r.outputs, want):
                    assert np.array_equal(bits(g), bits(w)), (name, n, params)
                if stats:
                    assert r.counters[abi.C_ADMITTED] == n
                    for c in WORK:
                        assert r.counters[c] == base.counters[c], (name, n, params, c)


def test_budget_holds_where_start_halts(gpu):
    """Every thread halts in START, so a wave refills until its input is gone
    and no other block runs: 40 STARTs a wave are over a budget of 8, and under
    one of 1000 they give the outputs and the counts of the compact form."""
    draw = started(1 << 15)
    want, _ = O.run("started_u64", draw)
    halts = np.flatnonzero(want[1] == 0)  # no other block ran
    rows = np.resize(halts, 40 * 256 * 64)
    ins, want = [a[rows] for a in draw], [w[rows] for w in want]

    def run(mode, **p):
        print(f"[gpu] all threads halt in START: mode {mode} {p}", flush=True)
        return loom_amd.run("started_u64", mode, ins, params=loom_amd.make_params(
            mode=mode, reconv=abi.RECONV_SWEEP, waves_per_cu=1, **p))

    with pytest.raises(abi.LoomError, match="0x2"):
        run(abi.MODE_HYBRID, max_steps=8)
    base = run(abi.MODE_COMPACT)
    for p in (dict(max_steps=1000), dict(), dict(stats=False), dict(refill=False)):
        r = run(abi.MODE_HYBRID, **p)
        for g, w in zip(r.outputs, want):
            assert np.array_equal(g, w), p
        for c in WORK:
            assert r.counters[c] == (base.counters[c] if p.get("stats", True) else 0), (p, c)


@pytest.mark.parametrize("stats", [True, False])
def test_jobs_share_a_pool(gpu, stats):
    """Jobs of two pooled kernels in one batch, one and many pools long: a
    wave that goes from one kernel's job to the other's uses the same LDS."""
    kernels = ("started_u64", "started_u32")
    for rows in ((1, 63, 64, 65, 129, 1000), (40000, 7, 30011, 500)):
        b, keep = loom_amd.Batch("start_mix"), []
        for i, n in enumerate(rows):
            for name in kernels:
                ins = [c.astype(dt) for c, dt in zip(started(n + i), loom_amd.kernel(name).inputs)]
                want, _ = O.run(name, ins)
                outs = [loom_amd.DeviceArray(n + i, dt) for dt in loom_amd.kernel(name).outputs]
                b.add(name, [loom_amd.DeviceArray.from_numpy(c) for c in ins], outs)
                keep.append((name, n + i, outs, want))
        for waves in (1, 0):
            print(f"[gpu] batch of pooled kernels {rows} stats {stats} waves {waves}", flush=True)
            b.run(loom_amd.make_params(mode=abi.MODE_HYBRID, stats=stats, waves_per_cu=waves))
            for name, n, outs, want in keep:
                for g, w in zip(outs, want):
                    assert np.array_equal(g.numpy(), w), (name, n, waves)
                    g.zero()
