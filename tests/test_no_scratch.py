"""No kernel of the library spills: the code objects' own metadata (private
segment and spilled registers of every kernel) in the built library."""
import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(path):
    """The gfx950 code objects of a library's offload bundles, one per translation unit."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, p)


def test_no_kernel_uses_scratch(tmp_path):
    readelf = next((p for p in ("/opt/rocm/llvm/bin/llvm-readelf", shutil.which("llvm-readelf")) if p and os.path.exists(p)), None)
    if not readelf:
        pytest.skip("llvm-readelf not found")
    from leap_amd.attention import load_library
    load_library()
    seen, spills = 0, {}
    for i, co in enumerate(_code_objects(os.path.join(ROOT, "leap_amd", "libleap_hip_attention.so"))):
        f = tmp_path / f"{i}.co"
        f.write_bytes(co)
        notes = subprocess.run([readelf, "--notes", str(f)], capture_output=True, text=True, check=True).stdout
        # a kernel's keys are sorted: .name, .private_segment_fixed_size, .vgpr_spill_count
        for m in re.finditer(r"\n    \.name: +(\S+)(.*?)\.wavefront_size", notes, re.S):
            seen += 1
            size = int(re.search(r"\.private_segment_fixed_size: +(\d+)", m.group(2)).group(1))
            spilled = int(re.search(r"\.vgpr_spill_count: +(\d+)", m.group(2)).group(1))
            if size or spilled:
                spills[m.group(1)] = (size, spilled)
    assert seen > 200, f"{seen} kernels found"
    assert not spills, spills
