"""The search writes its steps out over the slots of its row ring and counts ring rounds in the entries of its hash index, which it
clears when the count is used up: after 124 steps (two chunks of 1024 states to a compute unit, and merged kernels of 256 states
above 512 chunks: 93), 252 or 508, by the size of the index.  Chunk lengths around a ring's length and around the first and second
clearing, every size of the index, both layouts: steps that end a chunk anywhere in a round, and nothing else overwritten.  (That what is to be
cleared is cleared, test_search_index.py shows.)"""
import numpy as np
import pytest

from openfish_amd import synth
from oracle import crf_oracle as O
from test_gpu_merged import with_blank
from test_gpu_scan_options import api  # noqa: F401

pytestmark = pytest.mark.gpu

OPT = dict(q_scale=0.95, q_shift=-0.2)
# state_len, chunks, arrangement, steps between two clearings: a compute unit to a chunk, two and four chunks to a unit; merged kernels
SIZES = [(3, 2, 1, 508), (3, 170, 1, 252), (3, 516, 1, 124), (4, 2, 1, 508), (4, 514, 1, 124), (5, 2, 1, 508), (5, 130, 1, 93),
         (4, 2, 2, 252), (4, 514, 2, 93), (5, 2, 2, 252)]


@pytest.mark.parametrize("columns", [4, 5])
@pytest.mark.parametrize("state_len,N,arrangement,round_steps", SIZES)
def test_chunk_lengths_around_a_ring_and_around_a_clearing(api, state_len, N, arrangement, round_steps, columns):  # noqa: F811
    S = 4 ** state_len
    base = 2
    lengths = list(range(1, 10)) + [k * round_steps + d for k in ((1, 2) if round_steps < 508 else (1,)) for d in (-1, 0, 1, 2, 5)]
    longest = max(lengths)
    s16 = synth.crf_scores(longest, base, state_len, seed=11)
    gb = api.GpuBuf(longest, N, state_len)
    gb.set_split_scans(arrangement)
    for T in lengths:
        part = np.ascontiguousarray(s16[:T])
        ref = O.decode(part.astype(np.float32), state_len, OPT, nthreads=4)
        tiled = lambda a: np.concatenate([a] * (N // base))  # noqa: E731
        given = with_blank(part, T, base, S) if columns == 5 else part
        sc = api.upload_scores_to_hip(np.ascontiguousarray(np.tile(given, (1, N // base, 1))))
        mv, sq, _ = api.openfish_decode_gpu(T, N, columns * S, sc, state_len, api.DECODER_INIT(**OPT), gb)
        assert np.array_equal(mv, tiled(ref["moves"])), T
        assert np.array_equal(sq, tiled(ref["sequence"])), T
