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


@pytest.mark.parametrize("columns", [4, 5])
@pytest.mark.parametrize("state_len,T,N,enqueue", [(4, 1, 3, True), (4, 2, 1, True), (4, 37, 4, True), (4, 3, 513, True),
                                                   (4, 41, 515, True), (4, 5, 769, False), (5, 1, 16, False), (5, 2, 17, False),
                                                   (5, 38, 19, False)])
def test_forward_sweep_within_the_search_gives_the_oracle_s_tensors(api, state_len, T, N, enqueue, columns):
    """forward sweep and posterior in the beam search's workgroups, fed from its LDS rings; chunks shorter than the rings and batches that leave a workgroup half full"""
    S = 4 ** state_len
    s16 = synth.crf_scores(T, N, state_len, seed=T + N + state_len)
    given = s16
    if columns == 5:
        given = np.full((T, N, S, 5), np.nan, np.float16)
        given[..., 1:] = s16.reshape(T, N, S, 4)
        given = given.reshape(T, N, 5 * S)
    ref = O.decode(s16.astype(np.float32), state_len, {}, nthreads=8)
    sc = api.upload_scores_to_hip(given)
    gb = api.GpuBuf(T, N, state_len)
    gb.set_split_scans(api.SCANS_MERGED)
    api.lib().openfish_amd_memset(gb.handle.contents.post_NTC, 0xff, N * (T + 1) * S * 4)
    if enqueue:
        api.openfish_amd_decode_enqueue(T, N, columns * S, sc, state_len, api.DECODER_INIT(), gb)
        mv, sq, _ = api.openfish_amd_decode_wait(gb)
    else:
        mv, sq, _ = api.openfish_decode_gpu(T, N, columns * S, sc, state_len, api.DECODER_INIT(), gb)
    t = gb.timings()
    assert t["scan"] == 0 and t["path_sums"] == 0 and t["fwd_post"] > 0
    assert np.array_equal(gb.tensor("bwd_NTC"), ref["bwd"])
    close(gb.tensor("post_NTC"), ref["post"])
    assert np.array_equal(mv, ref["moves"]) and np.array_equal(sq, ref["sequence"])


# mean and spread of the scores, stay score, time steps: state values that hover about zero; that fall through negative
# powers of two; that rise past 2^19, where half an ulp is beyond what the proofs of estimates allow for; coarse ulps from the start
@pytest.mark.parametrize("mean,spread,stay,T", [(-1.65, 0.5, -1.65, 150), (-21.0, 3.0, -19.0, 220), (2600.0, 3.0, 2600.0, 230),
                                                (30000.0, 2000.0, 30000.0, 40), (-30000.0, 8.0, -30000.0, 40), (0.0, 12.0, 2.0, 120)])
@pytest.mark.parametrize("state_len,N", [(3, 3), (4, 2), (5, 1)])
def test_estimates_are_settled_right_at_every_magnitude(api, state_len, N, mean, spread, stay, T):  # noqa: F811
    """bwd bit for bit the oracle's, posteriors bit for bit those of the always-double arithmetic"""
    S = 4 ** state_len
    rng = np.random.default_rng(17 + T)
    s16 = np.clip(rng.normal(mean, spread, (T, N, 4 * S)), -65000, 65000).astype(np.float16)
    O.set_scan_stay(stay)
    try:
        ref_bwd, _, _ = O.scans(s16.astype(np.float32), state_len)
    finally:
        O.set_scan_stay()
    got = {}
    for fused in (False, True):
        for mode in ("two_tier", "precise"):
            bwd, post = stage_scans(api, s16, state_len, stay, api.SCAN_MODES[mode], fused)
            assert np.array_equal(bwd, ref_bwd), (fused, mode)
            got[fused, mode] = post
        assert np.array_equal(got[fused, "two_tier"], got[fused, "precise"], equal_nan=True)


@pytest.mark.parametrize("T,N", [(1, 256), (9, 255), (9, 257)])
@pytest.mark.parametrize("columns", [4, 5])
def test_backward_sweep_of_1024_states_on_either_side_of_a_chunk_per_unit(api, T, N, columns):  # noqa: F811
    four = synth.crf_scores(T, N, 5, seed=N + T)
    given = four
    if columns == 5:
        given = np.full((T, N, 1024, 5), np.nan, np.float16)
        given[..., 1:] = four.reshape(T, N, 1024, 4)
        given = given.reshape(T, N, 5 * 1024)
    ref_bwd, _, _ = O.scans(four.astype(np.float32), 5)
    bwd, _ = stage_scans(api, given, 5, 2.0, "two_tier", False)
    assert np.array_equal(bwd, ref_bwd)


MAGNITUDES = [(-1.65, 0.5, -1.65, 150), (-21.0, 3.0, -19.0, 220), (2600.0, 3.0, 2600.0, 230), (30000.0, 2000.0, 30000.0, 40),
              (-30000.0, 8.0, -30000.0, 40), (0.0, 12.0, 2.0, 120), (1.0, 0.2, 1.0, 300)]


# how a decode is made to take each form of the two-tier update: states per lane (several of them share a proof's trip),
# one kernel (four to a lane: one state after another, exponentials in a loop), sweep within the search, sweeps apart
@pytest.mark.parametrize("state_len,N,form", [(sl, n, (split, spl)) for sl, n in ((3, 3), (4, 2), (5, 1)) for split in (False, True) for spl in (0, 1, 2, 4)] +
                         [(4, 2, (2, 0)), (5, 2, (2, 0))])
@pytest.mark.parametrize("mean,spread,stay,T", MAGNITUDES)
def test_every_form_of_the_update_settles_estimates_right(api, state_len, N, form, mean, spread, stay, T):  # noqa: F811
    """bwd bit for bit the oracle's.  Posteriors are compared with those of the always-double arithmetic in the same number of
    kernels, which subtracts the same shift (another one would round the exponential's argument elsewhere: |x| 2^-24, 5e-6 for a
    posterior of 1e-31) but may take the normalising sums in another order: at most 3 + 6 + 8 additions of 2^-24 each way, a reciprocal
    of one ulp and a product, 2.5e-6 together.  A forward value that is an ulp off, |f| > 32, moves its posterior by
    3.8e-6 or more."""
    S = 4 ** state_len
    split, spl = form
    rng = np.random.default_rng(19 + T)
    s16 = np.clip(rng.normal(mean, spread, (T, N, 4 * S)), -65000, 65000).astype(np.float16)
    O.set_scan_stay(stay)
    try:
        ref_bwd, _, _ = O.scans(s16.astype(np.float32), state_len)
    finally:
        O.set_scan_stay()
    _, precise = stage_scans(api, s16, state_len, stay, api.SCAN_PRECISE, split is False)
    sc = api.upload_scores_to_hip(s16)
    gb = api.GpuBuf(T, N, state_len)
    gb.set_split_scans(split)
    gb.set_scan_states_per_lane(spl)
    api.lib().openfish_amd_memset(gb.handle.contents.post_NTC, 0xff, N * (T + 1) * S * 4)
    api.openfish_decode_gpu(T, N, 4 * S, sc, state_len, api.DECODER_INIT(blank_score=stay), gb)
    assert np.array_equal(gb.tensor("bwd_NTC"), ref_bwd)
    post = gb.tensor("post_NTC")
    finite = np.isfinite(precise)
    assert np.array_equal(np.isfinite(post), finite)
    np.testing.assert_allclose(post[finite], precise[finite], rtol=2.5e-6, atol=1.2e-38)
