"""The generations of the beam search's hash index wrap, and the search then clears it.  An entry that an element left behind
just one wrap ago, and that is still there, passes for a partner that is alive: the stay of the element's child is merged with a step
candidate it has nothing to do with, and that step is lost.

The inputs here bring this about in every event: a parent dies right after its child has been born, the child stays for one
wrap, and in the very step in which the parent's last entry would count again the child's true successor is born from the slot that
the parent had, with the child's own last base.  Guides (bwd) and scores are made up to say who lives: a stay adds 2, a step 0 where it is
meant and -8 elsewhere, and a guide of -60 ends a state.  A model of the index on the CPU, checked against the oracle, shows that without the clearing
the paths of all chunks change; the kernels have to give the oracle's, in every form of the index."""
import ctypes as C

import numpy as np
import pytest

from oracle import crf_oracle as O

# state_len, chunks, whether the forward sweep runs in the same kernel, index bits, steps between two clearings: a compute unit to a
# chunk, two and four chunks to a unit; merged with one and with two workgroups to a unit
FORMS = [(3, 16, False, 14, 508), (3, 170, False, 13, 252), (3, 516, False, 12, 124), (4, 16, False, 14, 508), (4, 72, False, 13, 252),
         (4, 514, False, 12, 124), (5, 16, False, 14, 508), (5, 40, False, 12, 93),
         (4, 18, True, 13, 252), (4, 514, True, 12, 93), (5, 16, True, 13, 252)]
UNIQUE = 16  # chunks that differ; a batch repeats them
STAY, CUT = 2.0, 100.0


def stalled(period, state_len, seed):
    """one chunk: scores [T][4S] and guides [T+1][S] of two stalls"""
    rng = np.random.default_rng(seed)
    S, T = 4 ** state_len, 2 * period + 45
    scores, bwd = np.full((T, 4 * S), -8.0, np.float16), np.zeros((T + 1, S), np.float32)
    step = lambda s, b: ((s << 2) & (S - 1)) | b  # noqa: E731

    def allow(t, s, to):  # the score of a step lies in the column of the base it drops
        scores[t, 4 * to + (s >> (2 * state_len - 2))] = 0.0

    root = int(rng.integers(S))
    bwd[0] = -60.0 - np.arange(S)  # the search begins with the 32 best
    bwd[1] = -60.0
    bwd[:2, root] = 0.0
    t = 2 + int(rng.integers(6))
    for _ in range(2):
        while True:
            b, y = rng.choice(4, 2, replace=False)
            child = step(root, int(b))
            after, other = step(child, int(b)), step(child, int(y))
            if len({root, child, after, other}) == 4:
                break
        allow(t, root, child)  # the child goes before the root: slots 0 and 1
        last = t + 2 + int(rng.integers(6))  # the root's last step, and its last entry in the index, as slot 1
        bwd[last + 1, root] = -60.0
        allow(last + 2 + int(rng.integers(4)), child, other)  # from here the child has slot 1
        allow(last + period, child, after)
        bwd[last + period + 2, [child, other]] = -60.0
        root = after
        t = last + period + 3 + int(rng.integers(4))
    assert t < T
    return scores, bwd


def batch(period, state_len):
    made = [stalled(period, state_len, 1000 * period + 10 * state_len + k) for k in range(UNIQUE)]
    return np.stack([m[0] for m in made], axis=1), np.stack([m[1] for m in made])


def model(scores, bwd, state_len, bits, period, clearing):
    """moves of one chunk by a search that finds partners through the index"""
    T, S = scores.shape[0], 4 ** state_len
    seed = lambda s: O.crc32c(0x12345678, s, 32)  # noqa: E731  (any hashes will do)
    root = int(np.argmax(bwd[0]))
    beam = [(seed(root), None, root, 0.0)]  # hash, hash of the sequence without its last base, state, score; the other 31 end in step 0
    slots, index, rows = (1 << bits) - 1, {}, []
    for t in range(T):
        if t % period == 0 and clearing:
            index.clear()
        for i, (h, _, _, _) in enumerate(beam):
            index[(h >> 2) & slots] = (h, t % period, i)
        intact = all(index[(h >> 2) & slots] == (h, t % period, i) for i, (h, _, _, _) in enumerate(beam))
        made = []
        for i, (h, _, s, sc) in enumerate(beam):
            for b in range(4):
                to = ((s << 2) & (S - 1)) | b
                made.append([(O.crc32c(h, b, 2), h, to), sc + float(scores[t, 4 * to + (s >> (2 * state_len - 2))]), i, 1])
        stays = [[(h, want, s), sc + STAY, i, 0] for i, (h, want, s, sc) in enumerate(beam)]
        for stay in stays:
            (_, want, s), _, _, _ = stay
            if want is None:
                continue
            if intact:
                h, gen, j = index.get((want >> 2) & slots, (None, None, 0))
                partner = j if h == want and gen == t % period and j < len(beam) else None
            else:
                partner = next((j for j, e in enumerate(beam) if e[0] == want), None)
            if partner is not None:
                other = made[4 * partner + (s & 3)]
                both = float(np.logaddexp(stay[1], other[1]))
                keep, lose = (stay, other) if stay[1] > other[1] else (other, stay)
                keep[1], lose[1] = both, -1e30
        made += stays
        guided = [m[1] + float(bwd[t + 1, m[0][2]]) for m in made]
        kept = [m for m, g in zip(made, guided) if g >= max(guided) - np.log(CUT)]
        assert 0 < len(kept) <= 25  # no further cut
        rows.append([(m[2], m[3]) for m in kept])
        best = max(range(len(kept)), key=lambda k: kept[k][1] + float(bwd[t + 1, kept[k][0][2]]))
        beam = [(m[0][0], m[0][1], m[0][2], m[1]) for m in kept]
    moves, at = np.zeros(T, np.uint8), best
    for t in reversed(range(T)):
        at, moves[t] = rows[t][at]
    moves[0] = 1
    return moves


def searched(scores, bwd, state_len):
    flat = np.full_like(bwd, 1.0 / bwd.shape[2])
    return O.decode_from_tensors(scores.astype(np.float32), state_len, bwd, flat, dict(blank_score=STAY, beam_cut=CUT), nthreads=4)


@pytest.mark.parametrize("state_len,bits,period", sorted({(f[0], f[3], f[4]) for f in FORMS}))
def test_an_entry_that_is_not_cleared_changes_the_path(state_len, bits, period):
    scores, bwd = batch(period, state_len)
    ref = searched(scores, bwd, state_len)
    for n in range(0, UNIQUE, 4):
        run = [model(scores[:, n], bwd[n], state_len, bits, period, clearing) for clearing in (True, False)]
        assert np.array_equal(run[0], ref["moves"][n]), n
        assert not np.array_equal(run[1], ref["moves"][n]), n


@pytest.fixture(scope="module")
def api():
    from openfish_amd import api as _api
    if _api.device_count() < 1:
        pytest.skip("no HIP device")
    return _api


@pytest.mark.gpu
@pytest.mark.parametrize("columns", [4, 5])
@pytest.mark.parametrize("state_len,N,merged,bits,period", FORMS)
def test_an_element_that_stays_for_a_wrap_finds_no_dead_partner(api, state_len, N, merged, bits, period, columns):
    S = 4 ** state_len
    scores, bwd = batch(period, state_len)
    ref = searched(scores, bwd, state_len)
    T, which = scores.shape[0], np.arange(N) % UNIQUE
    if columns == 5:
        four, scores = scores, np.full((T, UNIQUE, S, 5), np.nan, np.float16)
        scores[..., 1:] = four.reshape(T, UNIQUE, S, 4)
        scores = scores.reshape(T, UNIQUE, 5 * S)
    table = np.zeros(612)
    L = api.lib()
    L.openfish_amd_lse_table(table.ctypes.data_as(C.POINTER(C.c_double)))
    up = api.DeviceBuffer.from_host
    sc, bw, lse = up(scores[:, which]), up(bwd[which]), up(table)
    post, beam = api.DeviceBuffer(4 * N * (T + 1) * S), api.DeviceBuffer(64 * N * (T + 1))
    states, moves = api.DeviceBuffer(4 * N * T), api.DeviceBuffer(N * T)
    p, f = (lambda b: C.c_void_p(b.ptr)), C.c_float
    tail = (p(beam), p(states), p(moves), T, N, state_len, columns, f(np.log(np.float32(CUT))), f(STAY), p(lse), 0, None, None)
    if merged:
        assert L.ofk_beam_search_forward(p(sc), p(bw), p(post), *tail) == 0
    else:
        assert L.ofk_beam_search(p(sc), p(bw), *tail) == 0
    L.openfish_amd_sync()
    assert np.array_equal(moves.to_host(np.uint8, (N, T)), ref["moves"][which])
    assert np.array_equal(states.to_host(np.int32, (N, T)), ref["path_states"][which])
    for b in (sc, bw, lse, post, beam, states, moves):
        b.free()
