"""The forward sweep and the posterior within the beam search's kernel, asked for by the setter: its search under
the hooks that reach the serial merge replay and the colliding hashes, in every form of the kernel (256 states with
up to two and with up to four chunks on a compute unit, 1024 states), and the calls for which it does not exist."""
import numpy as np
import pytest

from openfish_amd import synth
from oracle import crf_oracle as O
from test_gpu_parity import qstring_close
from test_gpu_scan_options import api, close  # noqa: F401

pytestmark = pytest.mark.gpu

OPT = dict(q_scale=0.95, q_shift=-0.2)


def with_blank(s16, T, N, S):
    five = np.full((T, N, S, 5), np.nan, np.float16)
    five[..., 1:] = s16.reshape(T, N, S, 4)
    return five.reshape(T, N, 5 * S)


@pytest.mark.parametrize("columns", [4, 5])
@pytest.mark.parametrize("state_len,T,N,seed,copies", [(4, 240, 6, 2, 1), (4, 240, 6, 2, 86), (5, 90, 2, 4332, 1)])
def test_search_beside_the_forward_sweep_under_replay_and_colliding_hashes(api, state_len, T, N, seed, copies, columns):  # noqa: F811
    S = 4 ** state_len
    s16 = synth.crf_scores(T, N, state_len, seed=seed)
    plain = O.decode(s16.astype(np.float32), state_len, OPT, nthreads=4)
    O.set_seed_state_mask(15)
    try:
        collided = O.decode_from_tensors(s16.astype(np.float32), state_len, plain["bwd"], plain["post"], OPT, nthreads=4)
    finally:
        O.set_seed_state_mask()
    assert not np.array_equal(collided["moves"], plain["moves"])
    given = with_blank(s16, T, N, S) if columns == 5 else s16
    sc = api.upload_scores_to_hip(np.tile(given, (1, copies, 1)))  # above 512 chunks: four of them on a compute unit
    gb = api.GpuBuf(T, N * copies, state_len)
    gb.set_split_scans(api.SCANS_MERGED)
    for flags, ref in ((0, plain), (1, plain), (2, collided), (3, collided)):
        gb.set_debug_flags(flags)
        mv, sq, qs = api.openfish_decode_gpu(T, N * copies, columns * S, sc, state_len, api.DECODER_INIT(**OPT), gb)
        assert np.array_equal(mv, np.tile(ref["moves"], (copies, 1))), flags
        assert np.array_equal(sq, np.tile(ref["sequence"], (copies, 1))), flags
        qstring_close(qs, np.tile(ref["qstring"], (copies, 1)), mv)
    assert np.array_equal(gb.tensor("bwd_NTC"), np.tile(plain["bwd"], (copies, 1, 1)))
    close(gb.tensor("post_NTC"), np.tile(plain["post"], (copies, 1, 1)))


@pytest.mark.parametrize("state_len,mode,spl", [(3, "two_tier", 0), (4, "precise", 0), (4, "fast", 0), (5, "two_tier", 2)])
def test_asked_for_where_it_does_not_exist_another_arrangement_runs(api, state_len, mode, spl):  # noqa: F811
    T, N, S = 50, 3, 4 ** state_len
    s16 = synth.crf_scores(T, N, state_len, seed=9)
    sc = api.upload_scores_to_hip(s16)
    gb = api.GpuBuf(T, N, state_len)
    gb.set_scan_mode(mode)
    gb.set_scan_states_per_lane(spl)
    want = api.openfish_decode_gpu(T, N, 4 * S, sc, state_len, api.DECODER_INIT(**OPT), gb)
    gb.set_split_scans(api.SCANS_MERGED)
    got = api.openfish_decode_gpu(T, N, 4 * S, sc, state_len, api.DECODER_INIT(**OPT), gb)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
