"""Decodes that share the machine give, every time, the bytes of one that has it to itself: the search's waves of one batch
hold up those of the other's sweeps, which must not depend on who is quick."""
import numpy as np
import pytest

from openfish_amd import synth
from test_gpu_scan_options import api  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scans", [0, 1, 2])
@pytest.mark.parametrize("state_len,T,N", [(4, 1666, 256), (5, 400, 64)])
def test_batches_in_flight_repeat_the_bytes_of_one_alone(api, state_len, T, N, scans):  # noqa: F811
    S = 4 ** state_len
    inputs = [api.upload_scores_to_hip(synth.crf_scores(T, N, state_len, seed=70 + i, threads=8)) for i in range(2)]
    bufs = [api.GpuBuf(T, N, state_len) for _ in range(2)]
    opt = api.DECODER_INIT(q_scale=0.95, q_shift=-0.2)
    for gb in bufs:
        gb.set_split_scans(scans)
    want = [api.openfish_decode_gpu(T, N, 4 * S, x, state_len, opt, gb) for x, gb in zip(inputs, bufs)]
    bwd = [gb.tensor("bwd_NTC") for gb in bufs]
    for k in range(150):
        for x, gb in zip(inputs, bufs):
            api.openfish_amd_decode_enqueue(T, N, 4 * S, x, state_len, opt, gb)
        for gb, ref in zip(bufs, want):
            got = api.openfish_amd_decode_wait(gb)
            assert all(np.array_equal(a, b) for a, b in zip(got, ref)), k
    for gb, ref in zip(bufs, bwd):
        assert np.array_equal(gb.tensor("bwd_NTC"), ref)
