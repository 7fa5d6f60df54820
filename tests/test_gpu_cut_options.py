"""The cut-off of the beam search under every kind of beam_cut, on the kernels: none at all (zero, negative or infinite, which the losers of
merges pass), one that leaves a few or hardly any candidates, one that only the best pass (1), and
ones that the best itself does not pass (below 1), after which the beam is empty.  Scores as usual, scores of a few whole numbers and
constant ones: candidates that tie at the bounds, for which the bisection runs to its tenth guess and more than the beam's width are left.
Moves and bases are the oracle's, with every number of chunks to a workgroup and with the forward sweep in the search's workgroups."""
import numpy as np
import pytest

from openfish_amd import synth
from oracle import crf_oracle as O
from test_gpu_scan_options import api  # noqa: F401

pytestmark = pytest.mark.gpu

BASE, T = 4, 70
CUTS = [float("inf"), 3e38, 1e4, 17.0, 3.0, 1.5, 1.0, 0.999, 0.5, 1e-30, 0.0, -1.0]
# state_len, chunks, arrangement: a compute unit to a chunk, two and four chunks to a unit; merged, of 256 states two kernels
FORMS = [(3, 4, 1), (3, 300, 1), (3, 516, 1), (4, 4, 1), (4, 300, 1), (4, 516, 1), (5, 4, 1), (5, 132, 1), (4, 4, 2), (4, 516, 2), (5, 4, 2)]


def scores(kind, state_len):
    C = 4 ** (state_len + 1)
    if kind == "usual":
        return synth.crf_scores(T, BASE, state_len, seed=5, chunk_scale=np.array([0.05, 1.0, 2.5, 8.0], np.float32))
    if kind == "ties":
        rng = np.random.default_rng(6)
        return (rng.integers(0, 5, (T, BASE, C)) // np.array([1, 2, 3, 4])[None, :, None]).astype(np.float16)
    return np.broadcast_to(np.array([0.0, 2.0, -3.5, 60000.0], np.float16)[None, :, None], (T, BASE, C)).copy()


@pytest.mark.parametrize("kind", ["usual", "ties", "constant"])
@pytest.mark.parametrize("state_len,N,arrangement", FORMS)
def test_every_kind_of_cut_keeps_what_the_cpu_path_keeps(api, state_len, N, arrangement, kind):  # noqa: F811
    S = 4 ** state_len
    s16 = scores(kind, state_len)
    sc = api.upload_scores_to_hip(np.ascontiguousarray(np.tile(s16, (1, N // BASE, 1))))
    gb = api.GpuBuf(T, N, state_len)
    gb.set_split_scans(arrangement)
    for cut in CUTS:
        kw = dict(beam_cut=cut, q_scale=0.95, q_shift=-0.2)
        ref = O.decode(s16.astype(np.float32), state_len, kw, nthreads=4)
        mv, sq, _ = api.openfish_decode_gpu(T, N, 4 * S, sc, state_len, api.DECODER_INIT(**kw), gb)
        assert np.array_equal(mv, np.tile(ref["moves"], (N // BASE, 1))), cut
        assert np.array_equal(sq, np.tile(ref["sequence"], (N // BASE, 1))), cut
