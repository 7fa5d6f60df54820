"""The argument behind the halves that the beam search keeps of the cut-off's bounds (beam.hip), worked out here in exact fractions: the cuts
that come of them are the CPU path's (lo + hi) / 2, bit for bit, whichever way the bisection goes, at usual scores, next to zero and
next to the largest float.  This is arithmetic alone, no kernel runs: test_gpu_cut_options.py compares the kernels' cuts with the oracle's."""
from fractions import Fraction

import numpy as np
import pytest

F = np.float32
TOP = np.finfo(F).max


def rounded(x):
    """a fraction to the nearest float, ties to even"""
    near = F(float(x))
    return min((near, np.nextafter(near, F(-np.inf)), np.nextafter(near, F(np.inf))),
               key=lambda f: (abs(Fraction(float(f)) - x) if np.isfinite(f) else Fraction(10) ** 99, int(f.view(np.uint32)) & 1))


def fma(a, b, c):
    return rounded(Fraction(float(a)) * Fraction(float(b)) + Fraction(float(c)))


@pytest.mark.parametrize("scale", [1e-30, 1e-3, 1.0, 50.0, 4000.0, 1e6])
@pytest.mark.parametrize("log_cut", [4.6051702, 1e-4, 0.0, -0.7, 13.8, float(TOP)])
def test_cuts_from_halves_are_the_cpu_path_s(scale, log_cut):
    rng = np.random.default_rng(7)
    with np.errstate(over="ignore"):
        for _ in range(40):
            best = F(rng.normal() * scale)
            lo = cut_lo = np.maximum(best - F(log_cut), -TOP)
            hi = best
            half_lo, half_hi = F(0.5) * lo, F(0.5) * best
            want, got = (cut_lo + hi) / F(2), half_lo + half_hi
            assert got == want
            for guess in range(8):
                up, down = fma(got, 0.5, half_hi), fma(got, 0.5, half_lo)
                # below a cut at -max / 2 lie the losers of merges alone, of w elements w at most: fewer than 25 above it and more than 32 with
                # them cannot be, since w elements have 4 w candidates that lose nothing
                first_up = log_cut == float(TOP) and guess == 0
                assert up == (want + hi) / F(2) and (first_up or down == (lo + want) / F(2))
                half = F(0.5) * got
                if first_up or rng.random() < 0.5:
                    lo, half_lo, want, got = want, half, (want + hi) / F(2), up
                else:
                    hi, half_hi, want, got = want, half, (lo + want) / F(2), down
                assert F(2) * half_hi == hi
