"""Decodes of up to 96 chunks of 1024 states run the forward sweep beside the backward one, on compute units of its own, and take
the posteriors in a pass of their own (fwd_scan_kernel, posterior_rows_kernel in scan.hip).  Same tensors, bit for bit, as the
stages called one after another, and the backward ones as the CPU path's; at both sides of the limit, at lengths around
the rows kept in flight (6) and around a workgroup's share of the posterior's rows, peaked and flat chunks."""
import numpy as np
import pytest

from openfish_amd import synth
from oracle import crf_oracle as O
from test_gpu_merged import with_blank
from test_gpu_parity import close, gpu_scans
from test_gpu_scan_options import api  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("columns", [4, 5])
@pytest.mark.parametrize("T,N,stay", [(1, 1, 2.0), (2, 3, 2.0), (5, 2, 0.5), (6, 2, 2.0), (7, 5, 2.0), (11, 1, -1.5), (12, 43, 2.0), (13, 128, 2.0),
                                      (67, 96, 2.0), (67, 97, 2.0), (513, 1, 5.0), (300, 10, 2.0)])
def test_both_sweeps_at_once_leave_what_the_stages_leave(api, T, N, stay, columns):  # noqa: F811
    S = 1024
    base = min(N, 8)
    s16 = synth.crf_scores(T, base, 5, seed=T + N, chunk_scale=synth.stress_scale(base))
    s16 = np.ascontiguousarray(np.tile(s16, (1, -(-N // base), 1))[:, :N])
    given = with_blank(s16, T, N, S) if columns == 5 else s16
    sc = api.upload_scores_to_hip(given)
    gb = api.GpuBuf(T, N, 5)
    gb.set_split_scans(True)
    for _ in range(2):
        api.openfish_decode_gpu(T, N, columns * S, sc, 5, api.DECODER_INIT(q_scale=0.95, q_shift=-0.2, blank_score=stay), gb)
    bwd, post = gb.tensor("bwd_NTC"), gb.tensor("post_NTC")
    stage_bwd, stage_post = gpu_scans(api, given, 5, stay=stay)
    assert np.array_equal(bwd, stage_bwd)
    assert np.array_equal(post, stage_post)
    if stay == 2.0 and T < 100:
        ref = O.decode(s16[:, :base].astype(np.float32), 5, dict(q_scale=0.95, q_shift=-0.2), nthreads=4)
        assert np.array_equal(bwd[:base], ref["bwd"])
        close(post[:base], ref["post"], atol=1.2e-38)


def test_the_timings_tell_the_forward_sweep_from_the_posteriors_pass(api):  # noqa: F811
    T, N, S = 400, 8, 1024
    s16 = synth.crf_scores(T, N, 5, seed=3)
    sc, gb, opt = api.upload_scores_to_hip(s16), api.GpuBuf(T, N, 5), api.DECODER_INIT()
    gb.set_split_scans(True)
    for _ in range(2):
        api.openfish_decode_gpu(T, N, 4 * S, sc, 5, opt, gb)
    t = gb.timings()
    assert t["scan"] == 0 and 0 < t["fwd_post"] < t["fwd_scan"] < t["total"]  # a pass over rows against T dependent steps
    for change in (lambda: gb.set_scan_states_per_lane(2), lambda: gb.set_split_scans(False)):
        change()
        api.openfish_decode_gpu(T, N, 4 * S, sc, 5, opt, gb)
        assert gb.timings()["fwd_scan"] == 0
    gb.set_scan_states_per_lane(0)
    gb.set_split_scans(True)
    api.openfish_amd_decode_enqueue(T, N, 4 * S, sc, 5, opt, gb)  # may share the device: no units of its own
    api.openfish_amd_decode_wait(gb)
    assert gb.timings()["fwd_scan"] == 0 and gb.timings()["fwd_post"] > 0
