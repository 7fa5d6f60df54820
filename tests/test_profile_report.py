"""The report of a profile: how busy the device's vector units were, from counters as rocprofv3 writes them, and which kernel is which."""
import csv
import os
import subprocess
import sys

import pytest

from openfish_amd import profile_report as R

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CLOCKS = 4.9e6


def counters(path, kernel, values):
    os.makedirs(path)
    with open(os.path.join(path, "s_counter_collection.csv"), "w", newline="") as fh:
        out = csv.writer(fh)
        out.writerow(["Kernel_Name", "Counter_Name", "Counter_Value"])
        out.writerows([kernel, k, v] for k, v in values.items())


# 5 waves a SIMD are launched: all at once, or two rounds of half of them; a busy ALU all the time, or part of it
@pytest.mark.parametrize("resident,busy", [(5.0, 1.0), (2.5, 0.61), (2.5, 1.0), (0.3, 0.05)])
def test_waves_that_are_not_resident_at_once_do_not_count_as_if_they_were(tmp_path, resident, busy):
    kernel = "_ZN12_GLOBAL__N_111beam_kernelILi256ELi2ELi4ELi2EEEvPKDF16_"
    counters(tmp_path / "sq", kernel, {"SQ_WAVES": 5 * 1024, "SQ_BUSY_CYCLES": 32 * CLOCKS, "SQ_ACTIVE_INST_VALU": busy * 1024 * CLOCKS / 4})
    counters(tmp_path / "sq2", kernel, {"SQ_WAVE_CYCLES": resident * 1024 * CLOCKS / 4})
    text = subprocess.run([sys.executable, "-m", "openfish_amd.profile_report", str(tmp_path), "--title", "t", "--bench-args", "a"],
                          cwd=ROOT, capture_output=True, text=True, check=True).stdout
    head, = [line for line in text.splitlines() if "SIMD vector ALU busy |" in line]
    row = [line for line in text.splitlines() if line.startswith("| beam_kernel")][-1]
    cells = dict(zip((c.strip() for c in head.split("|")), (c.strip() for c in row.split("|"))))
    assert (cells["waves launched per SIMD"], cells["waves resident per SIMD"]) == ("5.00", "%.2f" % resident)
    assert cells["SIMD vector ALU busy"] == "%.2f" % busy


@pytest.mark.parametrize("name,short", [
    ("_ZN12_GLOBAL__N_115bwd_scan_kernelILi256ELi1ELi16ELi0ELb1EEEvPKDF16_Pfiifj", "bwd_scan_kernel<S=256,SPL=1,DEPTH=16,two_tier,early steps>"),
    ("void (anonymous namespace)::bwd_scan_kernel<256, 1, 16, 0, false>(_Float16 const*)", "bwd_scan_kernel<S=256,SPL=1,DEPTH=16,two_tier>"),
    ("void (anonymous namespace)::fwd_post_kernel<64, 1, 8, 0, true>(_Float16 const*)", "fwd_post_kernel<S=64,SPL=1,DEPTH=8,two_tier,early steps>"),
    ("_ZN12_GLOBAL__N_111beam_kernelILi64ELi1ELi5ELi0EEEvPKDF16_", "beam_kernel<S=64,chunks/group=1,columns=5>"),
])
def test_kernels_are_told_apart_by_all_their_parameters(name, short):
    assert R.short(name) == short
