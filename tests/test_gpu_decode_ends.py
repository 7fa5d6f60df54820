"""Where a decode's results come from and what its start and end are known by: the moves by a copy or, of small batches, by the
sequence stage; ends by events that the last kernels carry; a forward sweep on a lane of its own that has to wait for the null stream
where the scores are still on their way."""
import ctypes as C

import numpy as np
import pytest

from openfish_amd import synth
from test_gpu_scan_options import api  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("state_len,T,N", [(3, 2047, 64), (3, 2048, 64), (4, 1, 1), (4, 33, 3), (5, 8, 2)])
def test_moves_by_a_copy_and_by_the_sequence_stage_are_the_same(api, state_len, T, N):  # noqa: F811
    """64 chunks of 2048 steps are the first whose moves a blocking decode copies; those of enqueued ones the stage writes"""
    S = 4 ** state_len
    sc = api.upload_scores_to_hip(synth.crf_scores(T, N, state_len, seed=T + N))
    gb, opt = api.GpuBuf(T, N, state_len), api.DECODER_INIT(q_scale=0.95, q_shift=-0.2)
    for _ in range(3):
        blocking = [np.array(a) for a in api.openfish_decode_gpu(T, N, 4 * S, sc, state_len, opt, gb)]
        t = gb.timings()
        assert t["total"] >= t["beam"] > 0 and t["bwd"] >= 0 and t["scan"] >= 0
        assert np.array_equal(blocking[0], gb.tensor("moves"))
        api.openfish_amd_decode_enqueue(T, N, 4 * S, sc, state_len, opt, gb)
        assert all(np.array_equal(a, b) for a, b in zip(blocking, api.openfish_amd_decode_wait(gb)))


def test_both_sweeps_of_a_decode_wait_for_scores_that_are_still_on_their_way(api):  # noqa: F811
    """few chunks of 1024 states: the forward sweep starts beside the backward one, on another lane"""
    hip = api.lib()
    T, N, S = 60, 4, 1024
    old, new = (synth.crf_scores(T, N, 5, seed=s) for s in (21, 22))
    at, source = api.DeviceBuffer.from_host(old), api.DeviceBuffer.from_host(new)
    busy = [api.DeviceBuffer(1 << 28) for _ in range(2)]
    gb, opt = api.GpuBuf(T, N, 5), api.DECODER_INIT()
    api.openfish_decode_gpu(T, N, 4 * S, source.ptr, 5, opt, gb)
    assert gb.timings()["fwd_scan"] > 0
    want = gb.tensor("post_NTC")
    hip.hipDeviceSynchronize()
    for _ in range(80):
        assert hip.hipMemcpyAsync(C.c_void_p(busy[0].ptr), C.c_void_p(busy[1].ptr), C.c_size_t(1 << 28), 3, C.c_void_p()) == 0
    assert hip.hipMemcpyAsync(C.c_void_p(at.ptr), C.c_void_p(source.ptr), C.c_size_t(new.nbytes), 3, C.c_void_p()) == 0
    api.openfish_decode_gpu(T, N, 4 * S, at.ptr, 5, opt, gb)
    assert gb.timings()["fwd_scan"] > 0 and np.array_equal(gb.tensor("post_NTC"), want)
