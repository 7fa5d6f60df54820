"""bench.py's table of kernels: a kernel's time is set against the bytes that this kernel moves, in every arrangement of the scans."""
import pytest

import bench

# milliseconds of 37 chunks of 1024 states, T = 833, with both sweeps side by side and the posteriors' pass behind them
APART = {"scan": 0.0, "bwd": 0.667, "fwd_scan": 0.68, "fwd_post": 0.14, "beam": 0.49, "sequence": 0.022, "path_sums": 0.0, "total": 1.2}
SPLIT = dict(APART, fwd_scan=0.0, fwd_post=0.74)
T, N, S = 833, 37, 1024


def test_sweeps_apart_count_the_posterior_pass_by_itself():
    need = bench.algorithmic_bytes(5, T, N)
    vec = N * (T + 1) * S * 4
    scores = N * T * 4 * S * 2
    stages = bench.stage_table(need, APART, "split")
    assert stages["fwd_scan"]["algorithmic_GB"] == pytest.approx((scores + vec) / 1e9, abs=1e-4)
    assert stages["fwd_post"]["algorithmic_GB"] == pytest.approx(3 * vec / 1e9, abs=1e-4)
    beside = stages["beam_and_fwd_post_side_by_side"]
    assert beside["ms"] == 0.49 and beside["algorithmic_GB"] == pytest.approx((need["beam"] + 3 * vec) / 1e9, abs=1e-4)
    # from the start of the longer sweep to the end of the posteriors
    assert stages["scan_plus_posterior"]["ms"] == pytest.approx(0.68 + 0.14)
    assert bench.scans_text("split", APART) == bench.SCANS_TEXT["apart"]


def test_a_forward_kernel_with_its_posterior_keeps_its_bytes():
    need = bench.algorithmic_bytes(5, T, N)
    stages = bench.stage_table(need, SPLIT, "split")
    assert "fwd_scan" not in stages
    assert stages["fwd_post"]["algorithmic_GB"] == pytest.approx(need["fwd_post"] / 1e9, abs=1e-4)
    assert stages["scan_plus_posterior"]["ms"] == pytest.approx(0.667 + 0.74)
    merged = bench.stage_table(need, SPLIT, "merged")
    assert "fwd_post" not in merged and "scan_plus_posterior" not in merged
    assert merged["beam"]["algorithmic_GB"] == pytest.approx(need["beam_merged"] / 1e9, abs=1e-4)
