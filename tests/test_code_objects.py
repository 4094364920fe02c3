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
