"""What the compiler made of the kernels, read from the gfx950 code of the built library.

Registers that do not fit go to scratch memory, which inside a time step's loop costs more than the step.

The waves of a chunk exchange its state vector through LDS around a barrier, and a wave's writes have to be complete
before it passes: otherwise a wave that is quick reads the vector of two steps ago, which happens only while another
kernel's waves slow the writer down, and then to a few steps in a billion."""
import os
import re
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
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


def most_of(field, tmp_path):
    """the largest value of a field of the kernels' notes, by name (the scans are built twice, for both layouts of the scores)"""
    if not os.path.exists(READELF):
        pytest.skip("no llvm-readelf")
    blob = open(os.path.join(ROOT, "openfish_amd", "libopenfish_amd.so"), "rb").read()
    most = {}
    for i, code in enumerate(code_objects(blob)):
        path = tmp_path / ("%d.co" % i)
        path.write_bytes(code)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for kernel in re.split(r"\n\s+- \.agpr_count", notes)[1:]:
            name = re.search(r"\.name:\s+(\S+)", kernel).group(1)
            most[name] = max(most.get(name, 0), int(re.search(r"\.%s:\s+(\d+)" % field, kernel).group(1)))
    return most


def test_a_backward_sweep_finds_room_beside_another_decode_s_merged_kernel(tmp_path):
    """256 states, four columns: two chunks of the merged kernel are 14 waves on the four SIMDs of a unit, and a SIMD's 512 registers, given
    out by eights, are to hold four of them and a wave of the backward sweep, which keeps sixteen rows in flight"""
    registers = {k: (v + 7) // 8 * 8 for k, v in most_of("vgpr_count", tmp_path).items()}
    merged, = [v for k, v in registers.items() if "beam_kernelILi256ELi2ELi4ELi4E" in k]
    backward = [v for k, v in registers.items() if "bwd_scan_kernelILi256ELi1ELi16ELi0E" in k]
    assert len(backward) == 2 and 4 * merged + max(backward) <= 512, (merged, backward)  # with early steps and without


def test_no_kernel_keeps_registers_in_scratch(tmp_path):
    scratch = most_of("private_segment_fixed_size", tmp_path)
    assert any("scan_post_kernel" in k for k in scratch) and any("beam_kernel" in k for k in scratch)
    # both sweeps of 1024 states with four states to a lane keep a few values there between their phases
    allowed = {k: 32 for k in scratch if "scan_post_kernelILi1024ELi4E" in k}
    over = {k: v for k, v in scratch.items() if v > allowed.get(k, 0)}
    assert not over, over


def kernels(path):
    """(name, [(address, instruction, comment)]) of every function of a code object; llvm-objdump writes the target of a
    branch into the comment, as an offset from the function's start"""
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], capture_output=True, text=True, check=True).stdout
    name, code = None, []
    for line in text.splitlines():
        head = re.match(r"^[0-9a-f]+ <(.*)>:$", line)
        if head:
            if code:
                yield name, code
            name, code = head.group(1), []
            continue
        m = re.match(r"^\s+(\S.*?)\s*// ([0-9A-F]+):(.*)$", line)
        if m:
            code.append((int(m.group(2), 16), m.group(1), m.group(3)))
    if code:
        yield name, code


def barriers(code):
    """(number of barriers, those that some path reaches with an LDS operation of the wave not waited for)"""
    index = {address: i for i, (address, _, _) in enumerate(code)}
    after = []
    for i, (_, instruction, comment) in enumerate(code):
        op = instruction.split()[0]
        follow = [] if op in ("s_endpgm", "s_branch", "s_setpc_b64") else [i + 1] * (i + 1 < len(code))
        if op.startswith(("s_branch", "s_cbranch")):
            target = re.search(r"<[^>+]*(?:\+0x([0-9a-f]+))?>", comment)
            follow = follow + [index[code[0][0] + int(target.group(1) or "0", 16)]]
        after.append(follow)
    pending, todo, bad = [None] * len(code), [0], set()
    pending[0] = False
    while todo:
        i = todo.pop()
        instruction = code[i][1]
        state = pending[i]
        if instruction.startswith("s_barrier") and state:
            bad.add(i)
        if instruction.startswith("ds_"):
            state = True
        elif instruction.startswith("s_waitcnt") and "lgkmcnt(0)" in instruction:
            state = False
        for j in after[i]:
            if pending[j] is None or (state and not pending[j]):
                pending[j] = state
                todo.append(j)
    return sum(x[1].startswith("s_barrier") for x in code), sorted(bad)


def test_no_barrier_is_reached_with_an_lds_write_under_way(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    blob = open(os.path.join(ROOT, "openfish_amd", "libopenfish_amd.so"), "rb").read()
    seen, wrong = {}, []
    for i, code_object in enumerate(code_objects(blob)):
        path = tmp_path / ("%d.co" % i)
        path.write_bytes(code_object)
        for name, code in kernels(path):
            seen[name], bad = barriers(code)
            wrong += [(name, hex(code[b][0])) for b in bad]
    assert sum(n > 0 for k, n in seen.items() if "bwd_scan_kernel" in k or "scan_post_kernel" in k) >= 16, seen
    assert not wrong, wrong
