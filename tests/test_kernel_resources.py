"""Resources of the compiled kernels, from the metadata of the built library:
a spilled register is a round trip through memory on a path whose time is
memory."""
import os
import re
import struct
import subprocess

import pytest

from q36_amd import build

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _device_elfs(blob):
    """The gfx950 code objects of a library's offload bundles: after the magic
    the number of entries, then (offset, size, length of triple, triple) each,
    offsets from the magic on."""
    at = blob.find(MAGIC)
    while at >= 0:
        p = at + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", blob, p - 8)[0]):
            off, size, n = struct.unpack_from("<3Q", blob, p)
            triple = blob[p + 24:p + 24 + n]
            p += 24 + n
            if b"gfx950" in triple and size:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, at + len(MAGIC))


def test_no_kernel_uses_scratch(tmp_path):
    if not (os.path.exists(build.LIB) and os.path.exists(READELF)):
        pytest.skip("library or llvm-readelf absent")
    with open(build.LIB, "rb") as f:
        blob = f.read()
    kernels = {}
    for i, elf in enumerate(_device_elfs(blob)):
        p = tmp_path / f"{i}.elf"
        p.write_bytes(elf)
        notes = subprocess.run([READELF, "--notes", str(p)], capture_output=True, text=True, check=True).stdout
        for k in re.split(r"(?m)^ *- +\.agpr_count:", notes)[1:]:
            val = {m[0]: m[1] for m in re.findall(r"\.(name|private_segment_fixed_size|vgpr_spill_count): +(\S+)", k)}
            kernels[val["name"]] = int(val["private_segment_fixed_size"]), int(val["vgpr_spill_count"])
    assert any("k_direct_down" in n for n in kernels) and any("k_gateup_dma" in n for n in kernels)
    assert {n: v for n, v in kernels.items() if v != (0, 0)} == {}
