"""The scans at the edges of their pipelines: chunks shorter than the rows kept in flight, one step
either side of every multiple of them, groups of chunks that the batch does not fill.  The two-tier
arithmetic settles or resolves every update, so both arrangements must give the always-double bits
that the oracle gives."""
import numpy as np
import pytest

from openfish_amd import synth
from oracle import crf_oracle as O
from test_gpu_scan_options import api, close, stage_scans  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("state_len,N", [(3, 1), (3, 7), (4, 1), (4, 3), (5, 2)])
@pytest.mark.parametrize("columns", [4, 5])
def test_short_chunks(api, state_len, N, columns):  # noqa: F811
    S = 4 ** state_len
    for T in (1, 2, 3, 5, 7, 8, 9, 15, 16, 17, 31, 33):
        four = synth.crf_scores(T, N, state_len, seed=100 * T + N)
        ref = O.decode(four.astype(np.float32), state_len, {}, nthreads=4)
        s16 = four
        if columns == 5:
            s16 = np.full((T, N, S, 5), np.nan, np.float16)
            s16[..., 1:] = four.reshape(T, N, S, 4)
            s16 = s16.reshape(T, N, 5 * S)
        for fused in (False, True):
            bwd, post = stage_scans(api, s16, state_len, 2.0, "two_tier", fused)
            assert np.array_equal(bwd, ref["bwd"]), (T, fused)
            close(post, ref["post"])
