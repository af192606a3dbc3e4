"""No kernel of the built library keeps vector registers in memory (no GPU).

A spilled vector register is a trip to memory for each lane, and the tiles that
fill the register file have none to spare: three of them in the 256x256 tile's
epilogue cost 4096^3 half a percent.  The counts come from the metadata that the
compiler leaves in the code objects.
"""
import os
import re
import struct
import subprocess

import pytest

from fast_dl_amd import capi

READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(data):
    """The device code objects in a library's offload bundles."""
    at = data.find(MAGIC)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        entry = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, id_len = struct.unpack_from("<QQQ", data, entry)
            target = data[entry + 24:entry + 24 + id_len].decode()
            entry += 24 + id_len
            if target.startswith("hip") and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, entry)


@pytest.mark.skipif(not os.path.exists(READELF), reason="llvm-readelf not installed")
def test_no_kernel_spills_vector_registers(tmp_path):
    with open(capi.library_path(), "rb") as f:
        objects = list(code_objects(f.read()))
    spills = {}
    for i, code in enumerate(objects):
        path = tmp_path / f"code{i}.o"
        path.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True,
                               check=True).stdout
        names = re.findall(r"^    \.name: +(\S+)", notes, re.M)
        counts = [int(n) for n in re.findall(r"\.vgpr_spill_count: +(\d+)", notes)]
        assert len(names) == len(counts)
        spills.update(zip(names, counts))
    assert len(spills) > 200  # all of the GEMM's kernels were found
    assert {k: n for k, n in spills.items() if n} == {}
