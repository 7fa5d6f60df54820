"""What the compiler gave the kernels of the built library, from the metadata of its gfx950 code objects: registers that
do not fit go to scratch memory, which inside a time step's loop costs more than the step."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(blob):
    """gfx950 code objects of the offload bundles in a host library: after the magic a count, then per entry offset, size,
    length of the target's name and the name"""
    at = blob.find(BUNDLE)
    while at >= 0:
        count, = struct.unpack_from("<Q", blob, at + len(BUNDLE))
        p = at + len(BUNDLE) + 8
        for _ in range(count):
            offset, size, n = struct.unpack_from("<QQQ", blob, p)
            target = blob[p + 24:p + 24 + n].decode()
            p += 24 + n
            if "gfx950" in target and size:
                yield blob[at + offset:at + offset + size]
        at = blob.find(BUNDLE, at + 1)


def test_no_kernel_keeps_registers_in_scratch(tmp_path):
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    blob = open(os.path.join(ROOT, "openfish_amd", "libopenfish_amd.so"), "rb").read()
    scratch = {}
    for i, code in enumerate(code_objects(blob)):
        path = tmp_path / ("%d.co" % i)
        path.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for kernel in re.split(r"\n\s+- \.agpr_count", notes)[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel).group(1)
            used = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", kernel).group(1))
            scratch[name] = max(scratch.get(name, 0), used)
    assert any("scan_post_kernel" in k for k in scratch) and any("beam_kernel" in k for k in scratch)
    # both sweeps of 1024 states with four states to a lane keep a few values there between their phases
    allowed = {k: 32 for k in scratch if "scan_post_kernelILi1024ELi4E" in k}
    over = {k: v for k, v in scratch.items() if v > allowed.get(k, 0)}
    assert not over, over
