"""How many chunks of the beam search share a compute unit is chosen by their number and by whether the decode is alone on the
device (beam.hip, launch_beam): every form against the CPU path, at the sizes where the choice changes, under the hooks that
reach the comparison with all hashes, the serial merge replay and the colliding hashes."""
import numpy as np
import pytest

from openfish_amd import synth
from oracle import crf_oracle as O
from test_gpu_merged import OPT, with_blank
from test_gpu_parity import qstring_close
from test_gpu_scan_options import api  # noqa: F401

pytestmark = pytest.mark.gpu

# 64 and 256 states: a chunk per unit up to 64, alone 160; two up to 512; then four.  1024 states: up to 32, alone 128; then two
SIZES = [(3, 300, 8, n) for n in (8, 64, 65, 160, 161, 256, 257, 520)] + [(4, 240, 6, n) for n in (1, 64, 65, 160, 161, 256, 257)] + \
        [(5, 90, 2, n) for n in (2, 32, 33, 128, 129)]


@pytest.mark.parametrize("columns", [4, 5])
@pytest.mark.parametrize("state_len,T,base,N", SIZES)
def test_every_form_of_the_search_equals_the_cpu_path(api, state_len, T, base, N, columns):  # noqa: F811
    S = 4 ** state_len
    s16 = synth.crf_scores(T, base, state_len, seed=2 if state_len != 5 else 4332)
    s32 = s16.astype(np.float32)
    plain = O.decode(s32, state_len, OPT, nthreads=4)
    O.set_seed_state_mask(15)
    try:
        collided = O.decode_from_tensors(s32, state_len, plain["bwd"], plain["post"], OPT, nthreads=4)
    finally:
        O.set_seed_state_mask()
    many = -(-N // base)
    tiled = lambda a: np.concatenate([a] * many)[:N]  # noqa: E731
    sc = api.upload_scores_to_hip(np.ascontiguousarray(np.tile(with_blank(s16, T, base, S) if columns == 5 else s16, (1, many, 1))[:, :N]))
    bwd, post = api.DeviceBuffer.from_host(tiled(plain["bwd"])), api.DeviceBuffer.from_host(tiled(plain["post"]))
    opt, gb = api.DECODER_INIT(**OPT), api.GpuBuf(T, N, state_len)
    gb.set_split_scans(True)
    for flags, ref in ((0, plain), (1, plain), (2, collided), (3, collided)):
        gb.set_debug_flags(flags)
        for alone in (True, False):  # a blocking decode is; a search on tensors given to it may not be
            if alone:
                mv, sq, qs = api.openfish_decode_gpu(T, N, columns * S, sc, state_len, opt, gb)
            else:
                mv, sq, qs = api.openfish_amd_decode_from_tensors(T, N, columns * S, sc, state_len, opt, bwd, post, gb)
            assert np.array_equal(mv, tiled(ref["moves"])), (flags, alone)
            assert np.array_equal(sq, tiled(ref["sequence"])), (flags, alone)
            qstring_close(qs, tiled(ref["qstring"]), mv)
