"""What the host code refuses and what it asks of the runtime before a decode's first kernel: openfish_host.c against a HIP runtime
of two devices that executes nothing (host_stub.c), a process per case, because a refusal ends the process."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "openfish_amd", "csrc")

DRIVER = """
import ctypes as C, sys
L = C.CDLL(sys.argv[1])
L.openfish_gpubuf_init.restype = C.c_void_p
class Opt(C.Structure):
    _fields_ = [("w", C.c_size_t), ("f", C.c_float * 5), ("pad", C.c_bool)]
opt = Opt(32, (C.c_float * 5)(100.0, 2.0, 0.0, 1.0, 1.0), False)
T, N, SL = 8, 2, 3
scores = C.create_string_buffer(2 * T * N * 4 * 64)
tensor = C.create_string_buffer(4 * N * (T + 1) * 64)
busy = (C.c_int * 2).in_dll(L, "stub_null_busy")
out = [C.c_void_p() for _ in range(3)]
refs = [C.byref(p) for p in out]
def buf():
    return C.c_void_p(L.openfish_gpubuf_init(T, N, SL))
def decode(g):
    L.openfish_decode_gpu(T, N, 256, scores, SL, C.byref(opt), g, *refs)
def enqueue(g):
    L.openfish_amd_decode_enqueue(T, N, 256, scores, SL, C.byref(opt), g)
    L.openfish_amd_decode_wait(g, *refs)
def from_tensors(g):
    L.openfish_amd_decode_from_tensors(T, N, 256, scores, SL, C.byref(opt), tensor, tensor, g, *refs)
def seen(name):
    return C.c_int.in_dll(L, name).value
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "host.so")
    subprocess.check_call(["gcc", "-O1", "-shared", "-fPIC", "-std=gnu11", "-D__HIP_PLATFORM_AMD__", "-Wl,-Bsymbolic",
                           "-I", os.path.join(ROOT, "include"), "-I", CSRC, "-I", "/opt/rocm/include",
                           os.path.join(CSRC, "openfish_host.c"), os.path.join(ROOT, "tests", "host_stub.c"), "-o", so, "-lm", "-lpthread"])

    def go(code):
        return subprocess.run([sys.executable, "-c", DRIVER + code, so], capture_output=True, text=True)
    return go


CALLS = ["decode", "enqueue", "from_tensors"]


@pytest.mark.parametrize("busy", [0, 1])
@pytest.mark.parametrize("call", CALLS)
def test_a_decode_on_its_own_device_goes_through(run, call, busy):
    """and waits for the null stream where that has work left"""
    done = run("L.set_device_hip(1); g = buf(); busy[1] = %d; %s(g); print('joins', seen('stub_null_joins'))" % (busy, call))
    assert done.returncode == 0 and done.stdout == "joins %d\n" % busy, done


@pytest.mark.parametrize("busy", [0, 1])
@pytest.mark.parametrize("call", CALLS)
def test_a_gpubuf_of_another_device_is_refused(run, call, busy):
    """whatever the null stream of the present device is doing: it is not the one that the scores may still be on their way on"""
    done = run("g = buf(); L.set_device_hip(1); busy[0] = 1; busy[1] = %d; %s(g); print('went on')" % (busy, call))
    assert done.returncode == 1 and "went on" not in done.stdout, done


@pytest.mark.parametrize("busy", [0, 1])
@pytest.mark.parametrize("call", CALLS)
def test_an_error_that_the_caller_left_behind_is_still_reported(run, call, busy):
    """the launch of the kernel that was to make the scores, say: the first launch of the decode finds it"""
    done = run("g = buf(); busy[0] = %d; L.stub_fail(); %s(g); print('went on')" % (busy, call))
    assert done.returncode == 1 and "invalid configuration" in done.stderr and "went on" not in done.stdout, done


TIMED = """
T, N, SL = %d, %d, %d
scores = C.create_string_buffer(2 * T * N * 4 ** (SL + 1))
g = buf()
L.openfish_amd_gpubuf_set_split_scans(g, %d)
ms = (C.c_float * 8)()
def timed(intruder):
    C.c_int.in_dll(L, "stub_intruder").value = intruder
    L.openfish_decode_gpu(T, N, 4 ** (SL + 1), scores, SL, C.byref(opt), g, *refs)
    assert L.openfish_amd_last_timings(g, ms, 8) == 8
    print(*ms)
"""


# what the decode waits for on another lane: 64 states sweep and sums | sums; 256 states sweep | nothing but the copy of its moves | sums;
# few of 1024 states a sweep from the decode's start, and the posteriors' pass
@pytest.mark.parametrize("state_len,T,N,split,total", [(3, 8, 2, -1, 53), (3, 8, 2, 0, 52), (4, 8, 2, 1, 52), (4, 2048, 64, 2, 3), (4, 2048, 64, 0, 52),
                                                       (5, 20, 2, -1, 53)])
def test_a_decodes_times_begin_with_its_first_kernel_whatever_the_other_lanes_do(run, state_len, T, N, split, total):
    """another thread's decode puts 50 ms of work on every other stream while this one's kernels, a millisecond each, are being queued"""
    done = run(TIMED % (T, N, state_len, split) + "timed(50)")
    assert done.returncode == 0, done
    ms = dict(zip(("bwd", "fwd", "beam", "seq", "total", "scan", "sums", "fwd_scan"), map(float, done.stdout.split())))
    assert (ms["bwd"], ms["scan"]) == ((0, 1) if split == 0 else (1, 0)) and ms["beam"] == 1 and ms["seq"] == 1 and ms["total"] == total
    assert ms["fwd_scan"] == (51 if state_len == 5 else 0)


def test_a_forward_sweep_beside_the_backward_one_does_not_end_before_its_decode_starts(run):
    """decodes on lanes that are ahead of one another"""
    done = run(TIMED % (20, 2, 5, -1) + "for x in range(6): timed(50 - 7 * x)")
    assert done.returncode == 0, done
    for line in done.stdout.splitlines():
        bwd, fwd, beam, seq, total, scan, sums, fwd_scan = map(float, line.split())
        assert bwd == 1 and 1 <= fwd_scan < total, done.stdout
