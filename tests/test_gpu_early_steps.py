"""The sweeps take the double arithmetic at once while their values are small, in trips of eight steps (backward) and of the rows in
flight (forward), and go over to estimates where the values of a wave's lane 0 have passed a bound: chunks that end before, at and
behind that place, values that pass it in the first trip, late or never, waves of a chunk that pass it at different steps.  bwd bit for bit the
oracle's, posteriors within the bar of those of the always-double arithmetic."""
import numpy as np
import pytest

from oracle import crf_oracle as O
from test_gpu_scan_options import api, close, stage_scans  # noqa: F401

pytestmark = pytest.mark.gpu

# mean of the scores: values grow by that and about two; "uneven": a share of the states far ahead of the others
GROWTH = {"plain": 0.0, "fast": 45.0, "never": -3.6, "falling": -40.0, "uneven": 0.0}


def scores_of(kind, T, N, S, seed):
    rng = np.random.default_rng(seed)
    x = rng.normal(GROWTH[kind], 2.0, (T, N, S, 4))
    if kind == "uneven":  # reaching the first state of every second wave of either sweep costs or gives much
        x[:, :, ::128, :] += 300.0
        x[:, :, 64::128, :] -= 300.0
    return x.astype(np.float16).reshape(T, N, 4 * S)


@pytest.mark.parametrize("kind", sorted(GROWTH))
@pytest.mark.parametrize("state_len,N", [(3, 5), (3, 1025), (4, 2), (4, 257), (5, 1)])
def test_either_side_of_the_change(api, state_len, N, kind):  # noqa: F811
    S, stay = 4 ** state_len, -3.6 if kind == "never" else 2.0
    for T in (1, 7, 8, 9, 16, 17, 25, 41) if N > 99 else (1, 2, 7, 8, 9, 15, 16, 17, 24, 33, 64, 65, 137, 300):
        base = min(N, 3)
        s16 = scores_of(kind, T, base, S, 10 * T + N)
        O.set_scan_stay(stay)
        try:
            ref, _, _ = O.scans(s16.astype(np.float32), state_len)
        finally:
            O.set_scan_stay()
        tiled = np.ascontiguousarray(np.tile(s16, (1, -(-N // base), 1))[:, :N])
        bwd, post = stage_scans(api, tiled, state_len, stay, "two_tier", False)
        for n in (0, N // 2, N - 1):
            assert np.array_equal(bwd[n], ref[n % base]), (T, n)
        if N <= 99:
            _, precise = stage_scans(api, tiled, state_len, stay, "precise", False)
            close(post, precise)


@pytest.mark.parametrize("kind", sorted(GROWTH))
@pytest.mark.parametrize("T", [5, 18, 70, 160])
def test_both_sweeps_of_1024_states_apart(api, T, kind):  # noqa: F811
    """the forward recursion by itself: both sweeps at once against one behind the other"""
    s16 = scores_of(kind, T, 2, 1024, T)
    sc, opt = api.upload_scores_to_hip(s16), api.DECODER_INIT()
    got = []
    for split in (True, api.SCANS_MERGED):
        gb = api.GpuBuf(T, 2, 5)
        gb.set_split_scans(split)
        api.openfish_decode_gpu(T, 2, 4096, sc, 5, opt, gb)
        got.append((gb.tensor("bwd_NTC"), gb.tensor("post_NTC")))
        gb.free()
    assert np.array_equal(got[0][0], got[1][0])
    close(got[0][1], got[1][1])


@pytest.mark.parametrize("state_len,N,T", [(4, 256, 257), (4, 257, 256), (4, 257, 257), (3, 1024, 40), (3, 1025, 40)])
def test_either_side_of_the_sizes_that_have_early_steps(api, state_len, N, T):  # noqa: F811
    """kernels with and without them, bwd bit for bit the oracle's, posteriors within the bar of the always-double arithmetic's"""
    S = 4 ** state_len
    s16 = scores_of("plain", T, 3, S, N + T)
    ref, _, _ = O.scans(s16.astype(np.float32), state_len)
    tiled = np.ascontiguousarray(np.tile(s16, (1, -(-N // 3), 1))[:, :N])
    bwd, post = stage_scans(api, tiled, state_len, 2.0, "two_tier", False)
    _, precise = stage_scans(api, s16, state_len, 2.0, "precise", False)
    for n in (0, N // 2, N - 1):
        assert np.array_equal(bwd[n], ref[n % 3]), n
        close(post[n], precise[n % 3])
