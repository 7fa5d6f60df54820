"""The backward sweep keeps eight rows in flight instead of sixteen where more waves than four to a SIMD are asked for: either side of the
line, the same bits; and the same beside another decode's merged kernel as alone, whether or not that leaves compute units free."""
import numpy as np
import pytest

from openfish_amd import synth
from test_gpu_merged import with_blank
from test_gpu_scan_options import api  # noqa: F401

pytestmark = pytest.mark.gpu


def tiled_scores(T, N, state_len, columns, base=8):
    s16 = synth.crf_scores(T, base, state_len, seed=T + N)
    if columns == 5:
        s16 = with_blank(s16, T, base, 4 ** state_len)
    return np.ascontiguousarray(np.tile(s16, (1, -(-N // base), 1))[:, :N])


@pytest.mark.parametrize("columns", [4, 5])
@pytest.mark.parametrize("N", [384, 385, 512, 700])
@pytest.mark.parametrize("T", [7, 33])
def test_two_decodes_in_flight(api, T, N, columns):  # noqa: F811
    scores = tiled_scores(T, N, 4, columns)
    sc, opt = api.DeviceBuffer.from_host(scores), api.DECODER_INIT()
    call = (T, N, columns * 256, sc.ptr, 4, opt)
    alone = api.GpuBuf(T, N, 4)
    alone.set_split_scans(api.SCANS_MERGED)
    want = api.openfish_decode_gpu(*call, alone)
    bwd = alone.tensor("bwd_NTC")
    pair = [api.GpuBuf(T, N, 4) for _ in range(2)]
    for gb in pair:
        gb.set_split_scans(api.SCANS_MERGED)
        api.openfish_amd_decode_enqueue(*call, gb)
    for gb in pair:
        got = api.openfish_amd_decode_wait(gb)
        assert all(np.array_equal(a, b) for a, b in zip(got, want))
        assert np.array_equal(gb.tensor("bwd_NTC"), bwd)
    sc.free()


@pytest.mark.parametrize("state_len,N", [(4, 1024), (4, 1025), (3, 4096), (3, 4099)])
@pytest.mark.parametrize("T", [7, 33])
def test_one_state_to_a_lane_asked_for(api, state_len, N, T):  # noqa: F811
    scores = tiled_scores(T, N, state_len, 4)
    sc, opt = api.DeviceBuffer.from_host(scores), api.DECODER_INIT()
    bwd = []
    for spl in (1, 2):
        gb = api.GpuBuf(T, N, state_len)
        gb.set_split_scans(True)
        gb.set_scan_states_per_lane(spl)
        api.openfish_decode_gpu(T, N, 4 * 4 ** state_len, sc.ptr, state_len, opt, gb)
        bwd.append(gb.tensor("bwd_NTC"))
        gb.free()
    sc.free()
    assert np.array_equal(bwd[0], bwd[1])
