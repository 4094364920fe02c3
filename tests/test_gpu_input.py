"""How a hybrid run deals its input to the waves of its grid: dealt rounds,
guided claims from eight ranges, and the last batches of other ranges.  Every
thread must run exactly once at the sizes where the shares change: below and
around one batch per wave, four (claims begin), sixteen (other ranges are
tried) and a large remainder, on grids of one to several waves per CU and of
fewer waves than ranges, refilled, not refilled, with queues, and without
allocation."""
import ctypes as C

import numpy as np
import pytest

import loom_amd
from loom_amd import abi, workloads

pytestmark = pytest.mark.gpu

CUS = 256
FORMS = {
    "refill": dict(live_threshold=48),
    "refill at the last lane": dict(live_threshold=0),
    "no refill": dict(refill=False),
    "queues": dict(regroup=abi.REGROUP_QUEUES, live_threshold=32),
}


def fib(n):
    a, b, t = 0, 1, []
    for _ in range(91):
        t.append(a)
        a, b = b, a + b
    return np.array(t, np.uint64)[n.astype(np.int64)]


def check(n, wpc, stats, noalloc=False, **form):
    x = workloads.fib_inputs(n, seed=n)
    din = loom_amd.DeviceArray.from_numpy(x)
    out = loom_amd.DeviceArray.full(n, 0xFFFFFFFFFFFFFFFF, np.uint64)
    p = loom_amd.make_params(mode=abi.MODE_HYBRID, stats=stats, waves_per_cu=wpc, **form)
    if noalloc:
        st = abi.RunStats()
        ins, outs = (C.c_void_p * abi.MAX_IO)(din.ptr), (C.c_void_p * abi.MAX_IO)(out.ptr)
        abi.check(abi.load().loom_run_noalloc(loom_amd.kernel("fib_u64").index, abi.MODE_HYBRID,
                                              ins, outs, n, C.byref(p), C.byref(st)), "noalloc")
        admitted = st.counters[abi.C_ADMITTED]
    else:
        admitted = loom_amd.run("fib_u64", abi.MODE_HYBRID, [din], [out],
                                params=p).counters[abi.C_ADMITTED]
    assert np.array_equal(out.numpy(), fib(x)), (n, wpc, form)
    assert admitted == (n if stats else 0), (n, wpc, form)


@pytest.mark.parametrize("form", list(FORMS))
def test_every_thread_runs_once(gpu, form):
    wave = CUS * 64  # one batch for every wave of a grid of one wave per CU
    for n in (1, 64, 65, 64 * 7, 64 * 9 + 1, wave - 1, wave, wave + 1, 4 * wave - 1, 4 * wave,
              4 * wave + 64 * 9 + 5, 16 * wave - 63, 16 * wave, 16 * wave + 1, 41 * wave + 777):
        for wpc in (1, 3):
            print(f"[gpu] input {form} n={n} waves per CU {wpc}", flush=True)
            check(n, wpc, True, **FORMS[form])


def test_every_thread_runs_once_full_grid(gpu):
    for n in (1000003, 4 << 20, (8 << 20) + 12345):
        print(f"[gpu] input full grid n={n}", flush=True)
        check(n, 0, True, live_threshold=48)
        check(n, 0, False, live_threshold=48)
        check(n, 0, True, noalloc=True, live_threshold=48)
