"""The walk back through the beam slots, in blocks of 128 steps that up to four waves of a chunk deal round: at lengths around a block, around
as many blocks as waves and past them, in every form of the search (a chunk to a compute unit, two, four; with the forward sweep beside two
chunks, four, and one of 1024 states), against the oracle's moves and sequence."""
import numpy as np
import pytest

from openfish_amd import synth
from oracle import crf_oracle as O
from test_gpu_scan_options import api  # noqa: F401

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 127, 128, 129, 255, 256, 257, 385, 512, 513, 641, 1025]


@pytest.mark.parametrize("state_len,N,merged", [(3, 2, False), (3, 162, False), (3, 514, False), (4, 3, True), (4, 514, True), (5, 2, False), (5, 2, True),
                                                (5, 130, False)])
def test_paths_of_every_length_are_the_oracle_s(api, state_len, N, merged):  # noqa: F811
    S, base = 4 ** state_len, 2
    for T in LENGTHS if S < 1024 else [127, 129, 256, 257, 513]:
        s16 = synth.crf_scores(T, base, state_len, seed=T)
        ref = O.decode(s16.astype(np.float32), state_len, {}, nthreads=4, dump=False)
        sc = api.upload_scores_to_hip(np.ascontiguousarray(np.tile(s16, (1, -(-N // base), 1))[:, :N]))
        gb = api.GpuBuf(T, N, state_len)
        gb.set_split_scans(api.SCANS_MERGED if merged else True)
        mv, sq, _ = api.openfish_decode_gpu(T, N, 4 * S, sc, state_len, api.DECODER_INIT(), gb)
        for got, want in ((mv, ref["moves"]), (sq, ref["sequence"])):
            assert np.array_equal(got, np.tile(want, (-(-N // base), 1))[:N]), T
