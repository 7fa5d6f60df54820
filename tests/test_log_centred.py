"""The second tier's logarithm (openfish_amd/csrc/dmath.h, log_centred), host build, against long-double
libm over [1, 5], its cell picked with the sum itself and with an approximation on either side."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MAIN = r"""
#include "dmath.h"
#include <cstdio>
#include <cstdlib>
int main(int argc, char **argv) {
    static const double series[] = OFA_LOG_SERIES;
    ofa::LogCell cells[ofa::kLogCentredCells];
    for (int i = 0; i < ofa::kLogCentredCells; ++i) cells[i] = ofa::log_centred_cell(i);
    const int away = atoi(argv[1]);  // ulps between the sum and its approximation
    double worst = 0;
    for (uint32_t b = 0x3f800000u; b <= 0x40a00000u; b += 5) {
        const uint32_t near = b + (uint32_t)away < 0x3f800000u ? 0x3f800000u : b + (uint32_t)away;
        const float s = ofa::float_of(b);
        const double got = ofa::log_centred(s, cells[ofa::log_centred_index(ofa::float_of(near))], series);
        const double err = (double)fabsl((long double)got - logl((long double)s));
        worst = err > worst ? err : worst;
    }
    printf("%.17g %.17g\n", worst, ofa::log_centred(1.0f, cells[ofa::log_centred_index(1.0f)], series));
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("log_centred")
    (d / "main.cpp").write_text(MAIN)
    subprocess.check_call(["g++", "-O2", "-ffp-contract=off", "-I", os.path.join(ROOT, "openfish_amd", "csrc"),
                           str(d / "main.cpp"), "-o", str(d / "main"), "-lm"])
    return str(d / "main")


@pytest.mark.parametrize("away", [0, 16, -16])
def test_log_centred(exe, away):
    worst, ln1 = map(float, subprocess.check_output([exe, str(away)]).split())
    assert worst < 2.0 ** -51
    assert ln1 == 0.0
