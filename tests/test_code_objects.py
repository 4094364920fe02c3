"""Resources of the device kernels that the library holds, from the metadata of
its gfx950 code objects: what a kernel is compiled to without being asked for
(scratch, LDS) is a cost that no result shows."""
import re
import shutil
import struct
import subprocess

import pytest

from loom_amd import build

READELF = shutil.which("llvm-readelf", path="/opt/rocm/llvm/bin") or shutil.which("llvm-readelf")
EM_AMDGPU = 224


def code_objects(path):
    """The AMDGPU ELF images in the fat binaries of a library."""
    data = path.read_bytes()
    at = data.find(b"\x7fELF", 4)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == EM_AMDGPU:
            # its section headers are the last of it
            shoff, = struct.unpack_from("<Q", data, at + 0x28)
            size, count = struct.unpack_from("<HH", data, at + 0x3A)
            yield data[at:at + shoff + size * count]
        at = data.find(b"\x7fELF", at + 4)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """(mangled name, its metadata) of every kernel."""
    if READELF is None:
        pytest.skip("no llvm-readelf")
    found = []
    for i, image in enumerate(code_objects(build.LIB)):
        f = tmp_path_factory.mktemp("co") / f"{i}.elf"
        f.write_bytes(image)
        notes = subprocess.run([READELF, "--notes", str(f)], capture_output=True, text=True,
                               check=True).stdout
        for part in notes.split("- .agpr_count:")[1:]:
            keys = dict(re.findall(r"^ +\.(\w+): +(\S+)$", part, re.M))
            found.append((keys["name"], {k: int(v) for k, v in keys.items() if v.isdigit()}))
    assert len(found) > 100
    return found


def test_batch_kernels_use_no_scratch(kernels):
    """Under any policy: an occupancy hint measured under one of them must not
    cost the others their registers."""
    batch = [(n, m) for n, m in kernels if "12batch_kernelI" in n]
    assert {re.search(r"batch_kernelILi(\d)", n).group(1) for n, _ in batch} == {"0", "1", "2"}
    spilled = {n[:60]: m["private_segment_fixed_size"] for n, m in batch
               if m["private_segment_fixed_size"]}
    assert not spilled


def one_wave(kernels, name):
    """The sweeping kernels of one-wave workgroups that may hold a pool of
    started threads: (mangled name, metadata)."""
    return [(n, m) for n, m in kernels if re.search(name, n)]


def lds_waves(m):
    """Waves of a SIMD that a CU's 160 KB in granules of 1280 bytes hold."""
    return 160 * 1024 // max(1280, -(-m["group_segment_fixed_size"] // 1280) * 1280) // 4


def test_pool_costs_no_waves(kernels):
    """A pool of started threads takes no more LDS than its kernel's registers
    leave waves for, however much is live after START."""
    pooled = one_wave(kernels, r"18hybrid_pass_kernelI.*Li2ELb0ELb.E|12batch_kernelILi2E")
    assert len(pooled) > 20
    fewer = {}
    for n, m in pooled:
        by_registers = min(8, 512 // (-(-m["vgpr_count"] // 8) * 8))
        if lds_waves(m) < by_registers:
            fewer[n[-80:]] = (m["group_segment_fixed_size"], m["vgpr_count"])
    assert not fewer


def test_members_of_a_batch_share_a_pool(kernels):
    """The batch kernel of two pooled kernels has the larger one's pool, and
    both lookup tables."""
    started = {n: m["group_segment_fixed_size"] for n, m in kernels
               if "115ELc116ELc97ELc114ELc116ELc101ELc100E" in n}  # "started"
    of = {t: max(v for n, v in started.items() if re.search(
        rf"18hybrid_pass_kernelI.*8VariableI{t}.*Li2ELb0ELb.E", n)) for t in "jm"}
    batch = [v for n, v in started.items() if "12batch_kernelILi2E" in n]
    table = 32  # of a jump of four targets, aligned
    assert len(batch) == 2 and max(batch) <= max(of.values()) + table
    assert min(of.values()) > 1024
