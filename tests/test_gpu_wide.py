"""Straight-line kernels of narrow columns, several threads per lane (large runs
without statistics): every output equals the oracle's bit for bit at the sizes
where the lane's share is cut off, and over columns that are not aligned for
it, which take the general kernel."""
import numpy as np
import pytest

import loom_amd
from loom_amd import abi, workloads
from tests import oracle_lib as O

pytestmark = pytest.mark.gpu

LARGE = 4 << 20  # threads from which lanes take four


def words(n, seed):
    return np.random.default_rng(seed).integers(0, 1 << 32, n, dtype=np.uint32)


INPUTS = {
    "threefry2x32_u32": workloads.threefry_inputs,
    "fp_mix_f32": lambda n: [np.random.default_rng(3).uniform(-900, 900, n).astype(np.float32),
                             np.random.default_rng(4).uniform(-900, 900, n).astype(np.float32)],
    "int_mix_u32": lambda n: [words(n, 5), words(n, 6)],
    "sct_range_f32": lambda n: [words(n, 7) % np.uint32(9)],
    "roots_f32": lambda n: [words(n, 8).view(np.float32)],
}


class Shifted(loom_amd.DeviceArray):
    """A column that begins `by` elements after its allocation."""

    def __init__(self, n, dtype, by):
        self.whole = loom_amd.DeviceArray(n + by, dtype)
        self.dtype, self.n = np.dtype(dtype), n
        self.nbytes = n * self.dtype.itemsize
        self.ptr = self.whole.ptr + by * self.dtype.itemsize

    def free(self):
        pass


def same(g, w):
    nan = np.isnan(g) & np.isnan(w) if g.dtype.kind == "f" else np.zeros(len(g), bool)
    return ((g.view(np.uint32) == w.view(np.uint32)) | nan).all()


@pytest.mark.parametrize("name", list(INPUTS))
def test_wide_matches_oracle(gpu, name):
    k = loom_amd.kernel(name)
    ins = INPUTS[name](LARGE + 1029)
    want, _ = O.run(name, ins)
    for n, by in ((LARGE - 1, 0), (LARGE, 0), (LARGE + 1, 0), (LARGE + 3, 0), (LARGE + 1029, 0),
                  (LARGE + 3, 1), (LARGE + 3, 2)):
        print(f"[gpu] wide {name} n={n} columns shifted by {by}", flush=True)
        din = []
        for a in ins:
            col = Shifted(n, a.dtype, by)
            cut = np.ascontiguousarray(a[:n])
            abi.check(abi.load().loom_memcpy_h2d(col.ptr, cut.ctypes.data, cut.nbytes), "h2d")
            din.append(col)
        out = [Shifted(n + 8, dt, by) for dt in k.outputs]
        for o in out:
            o.zero()
        loom_amd.run(k, abi.MODE_COMPACT, din, out, n=n,
                     params=loom_amd.make_params(stats=False))
        for o, w in zip(out, want):
            g = o.numpy()
            assert same(g[:n], w[:n]), (name, n, by)
            assert not g[n:].view(np.uint32).any(), (name, n, by)
