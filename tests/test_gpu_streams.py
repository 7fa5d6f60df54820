"""The streams of the gpubufs: whichever hardware queues the runtime deals them to, a split decode has to run its
forward sweep beside the beam search, and two batches in flight have to run side by side, with one gpubuf in the
process and with several."""
import threading
import time

import numpy as np
import pytest

from openfish_amd import synth
from test_gpu_parity import qstring_close
from test_gpu_scan_options import api  # noqa: F401

pytestmark = pytest.mark.gpu

STATE_LEN, T, N = 4, 1000, 64
S = 4 ** STATE_LEN


@pytest.fixture(scope="module")
def scores(api):  # noqa: F811
    return api.upload_scores_to_hip(synth.crf_scores(T, N, STATE_LEN, seed=3))


def test_forward_sweep_runs_beside_the_search_in_every_gpubuf(api, scores):  # noqa: F811
    """64 chunks of 256 states leave nine tenths of the machine idle: the forward sweep takes 0.8 of the search's time
    beside it, and ends 1.7 times that time after the backward sweep where it has to wait for the search"""
    bufs, ratios = [], []
    for _ in range(7):
        gb = api.GpuBuf(T, N, STATE_LEN)
        gb.set_split_scans(True)
        bufs.append(gb)  # kept: streams of its own would find the queues shared by more each time
        seen = []
        for _ in range(3):
            api.openfish_decode_gpu_discard(T, N, 4 * S, scores, STATE_LEN, api.DECODER_INIT(), gb)
            t = gb.timings()
            seen.append(t["fwd_post"] / t["beam"])
        ratios.append(min(seen))
    assert max(ratios) < 1.25, ratios


@pytest.mark.parametrize("batches,others", [(2, 0), (2, 1), (2, 2), (2, 3), (3, 0), (3, 1)])
def test_batches_in_flight_run_side_by_side(api, scores, batches, others):  # noqa: F811
    """two or three decodes of 64 chunks together take 1.1 to 1.2 times as long as one, and twice as long where two of them
    share a queue or one sits in the null stream's"""
    kept = [api.GpuBuf(32, 1, 3) for _ in range(others)]
    bufs = [api.GpuBuf(T, N, STATE_LEN) for _ in range(batches)]

    def ms(which):
        best = 1e9
        for _ in range(5):
            t0 = time.perf_counter()
            for gb in which:
                api.openfish_amd_decode_enqueue(T, N, 4 * S, scores, STATE_LEN, api.DECODER_INIT(), gb)
            for gb in which:
                api.openfish_amd_decode_wait(gb, copy=False)
            best = min(best, time.perf_counter() - t0)
        return best * 1e3

    ms(bufs)
    one, together = ms(bufs[:1]), ms(bufs)
    assert together < 1.6 * one, (one, together)
    del kept


def test_gpubufs_made_used_and_freed_by_several_threads(api, scores):  # noqa: F811
    """the streams that gpubufs share come and go with them: threads that make, use and free gpubufs at the same time, down to
    none and up again, all get the results of a single one (the quality characters within their bound: a decode that finds
    another under way takes another arrangement, whose posteriors are summed in another order)"""
    def decode():
        gb = api.GpuBuf(T, N, STATE_LEN)
        out = api.openfish_decode_gpu(T, N, 4 * S, scores, STATE_LEN, api.DECODER_INIT(), gb)
        gb.free()
        return out

    want, wrong = decode(), []

    def work():
        api.lib().set_device_hip(0)
        for _ in range(5):
            try:
                mv, sq, qs = decode()
                assert np.array_equal(mv, want[0]) and np.array_equal(sq, want[1])
                qstring_close(qs, want[2], mv)
            except Exception as e:  # an exception in a thread would otherwise pass silently
                wrong.append(e)

    threads = [threading.Thread(target=work) for _ in range(3)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not wrong, wrong
