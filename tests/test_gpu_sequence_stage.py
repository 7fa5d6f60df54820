"""The sequence stage takes base positions from running sums over pieces of 64 time steps, gathers with all waves but one, and moves
the characters of a chunk, which begin at any address, in pieces of 16 bytes (sequence.hip): lengths around all of these, one
workgroup size each side of 256 chunks, chunks that are all moves and chunks that have hardly any.  Fed the CPU path's tensors
the bytes are the CPU path's; an enqueued decode writes its moves from the same kernel."""
import numpy as np
import pytest

from openfish_amd import synth
from oracle import crf_oracle as O
from test_gpu_parity import gpu_from_tensors, qstring_close
from test_gpu_scan_options import api  # noqa: F401

pytestmark = pytest.mark.gpu

LENGTHS = (1, 2, 15, 16, 17, 63, 64, 65, 447, 448, 449, 959, 960, 961, 1025, 4095, 4096, 4097, 4160, 4161, 8191, 8192)
SHAPES = [(3, T, 3) for T in LENGTHS] + [(4, 461, 5), (5, 131, 3)] + \
         [(sl, T, N) for sl, T in ((3, 67), (4, 33)) for N in (256, 257)] + [(3, 449, 300), (5, 18, 258)]


@pytest.mark.parametrize("state_len,T,N", SHAPES)
def test_bytes_are_the_cpu_paths(api, state_len, T, N):  # noqa: F811
    base = min(N, 4)
    s16 = synth.crf_scores(T, base, state_len, seed=3 * T + N, chunk_scale=synth.stress_scale(base))
    many = -(-N // base)
    tiled = lambda a: np.concatenate([a] * many)[:N]  # noqa: E731
    given = np.ascontiguousarray(np.tile(s16, (1, many, 1))[:, :N])
    for blank in (2.0, -60.0, 60.0):
        kw = dict(q_scale=0.95, q_shift=-0.2, blank_score=blank)
        ref = O.decode(s16.astype(np.float32), state_len, kw, nthreads=4)
        (mv, sq, qs), gb = gpu_from_tensors(api, given, state_len, kw, tiled(ref["bwd"]), tiled(ref["post"]))
        assert np.array_equal(mv, tiled(ref["moves"])), blank
        assert np.array_equal(sq, tiled(ref["sequence"])), blank
        assert np.array_equal(qs, tiled(ref["qstring"])), blank
        assert np.array_equal(gb.tensor("states"), tiled(ref["states"])), blank


@pytest.mark.parametrize("T,N", [(T, N) for T in (1, 17, 65, 449, 961) for N in (3, 257)])
def test_an_enqueued_decode_writes_the_same_bytes(api, T, N):  # noqa: F811
    base = min(N, 4)
    s16 = synth.crf_scores(T, base, 3, seed=T, chunk_scale=synth.stress_scale(base))
    ref = O.decode(s16.astype(np.float32), 3, dict(q_scale=0.95, q_shift=-0.2), nthreads=4)
    many = -(-N // base)
    tiled = lambda a: np.concatenate([a] * many)[:N]  # noqa: E731
    sc = api.upload_scores_to_hip(np.ascontiguousarray(np.tile(s16, (1, many, 1))[:, :N]))
    gb, opt = api.GpuBuf(T, N, 3), api.DECODER_INIT(q_scale=0.95, q_shift=-0.2)
    for _ in range(2):
        api.openfish_amd_decode_enqueue(T, N, 4 * 64, sc, 3, opt, gb)
        mv, sq, qs = api.openfish_amd_decode_wait(gb)
        assert np.array_equal(mv, tiled(ref["moves"]))
        assert np.array_equal(sq, tiled(ref["sequence"]))
        qstring_close(qs, tiled(ref["qstring"]), mv)
