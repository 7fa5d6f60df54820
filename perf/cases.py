"""The work that users of this library have it do, as cases that can be timed.

A basecaller hands over one batch of CRF scores per network run (fp16, time step by chunk by state, four
or five columns per state) and gets moves, bases and qualities back in host memory: `decode` is the
blocking call, `flight` the same through enqueue and wait with a batch on each of two gpubufs.  `rotary`
is the in-place rotary embedding that the transformer models call on a layer's queries and keys.

Models are told apart by state_len: 3, 4 and 5 (64, 256 and 1024 states: the fast, hac and sup
configurations of bench.py).  Chunks are 1666 time steps long in these configurations; 833 are those of a
model with twice the stride, and the end of a run brings shorter chunks and batches that are not full.
"""
import math

import torch

from openfish_amd import api, synth

# q_scale, q_shift per model, as bench.py decodes with
QUALITY = {3: (0.97, -1.8), 4: (0.95, -0.2), 5: (0.95, 0.5)}
MOST_STATES = 1024 * 1666 * 256  # chunks x time steps x states of the largest batch


def _decode(name, state_len, T, N, columns, mix="plain", op="decode"):
    return {"name": name, "op": op, "state_len": state_len, "T": T, "N": N, "columns": columns, "mix": mix}


def _rotary(name, batch, seqlen, nheads, head_dim, half):
    return {"name": name, "op": "rotary", "batch": batch, "seqlen": seqlen, "nheads": nheads, "head_dim": head_dim,
            "half": half}


def listed():
    return [
        # a single read's tail: short chunks, few of them, the call's own cost counts
        _decode("hac_n5_t96", 4, 96, 5, 4),
        # one chunk, as in the known-answer test of the command-line driver
        _decode("fast_n1", 3, 1666, 1, 4),
        # a small batch of the smallest model
        _decode("fast_n16", 3, 1666, 16, 5),
        # a part-filled batch of the largest model, half-length chunks
        _decode("sup_n37_t833", 5, 833, 37, 4),
        # ragged in both directions, blank column kept
        _decode("hac_n403_t1201", 4, 1201, 403, 5),
        # the full batch of every model
        _decode("fast_n512", 3, 1666, 512, 5),
        _decode("hac_n512", 4, 1666, 512, 4),
        _decode("sup_n256", 5, 1666, 256, 5),
        # the largest batch; half of the chunks peaked, half nearly uniform
        _decode("hac_n1024_stress", 4, 1666, 1024, 5, "stress"),
        # a caller that keeps two batches in flight
        _decode("hac_n512_flight", 4, 1666, 512, 4, op="flight"),
        # rotary embedding of one short sequence, and of a full batch
        _rotary("rotary_b2_l33", 2, 33, 8, 64, 32),
        _rotary("rotary_b500_l833", 500, 833, 8, 64, 32),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.25:
        half = rng.choice((32, 32, 16, 8, 64, 12))  # 12: pairs that do not come in eights
        nheads = rng.choice((1, 3, 4, 8, 12))
        seqlen = _log_int(rng, 16, 1700)
        most = 500 * 833 * 512 // (seqlen * nheads * 2 * half)
        return {k: v for k, v in _rotary("", _log_int(rng, 1, max(1, min(500, most))), seqlen, nheads, 2 * half,
                                         half).items() if k != "name"}
    op = "flight" if rng.random() < 0.15 else "decode"
    state_len = rng.choice((3, 4, 5))
    T = _log_int(rng, 32, 2000)
    most = MOST_STATES // (T * 4 ** state_len) // (2 if op == "flight" else 1)
    N = _log_int(rng, 1, max(1, min(1024, most)))
    made = _decode("", state_len, T, N, rng.choice((4, 5)), rng.choice(("plain", "plain", "stress")), op)
    return {k: v for k, v in made.items() if k != "name"}


def _scores(case, gen):
    """N(0, 2) scores, the blank column one higher (synth.crf_scores' description of a CRF head, drawn on
    the GPU); `stress` scales even chunks by 6 and odd ones by 0.2"""
    T, N, S, cols = case["T"], case["N"], 4 ** case["state_len"], case["columns"]
    x = torch.empty((T, N, S, cols), dtype=torch.float16, device="cuda").normal_(0.0, 2.0, generator=gen)
    if case["mix"] == "stress":
        x *= torch.from_numpy(synth.stress_scale(N)).cuda().half()[None, :, None, None]
    if cols == 5:
        x[..., 0] += 1.0
    return x


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    if case["op"] == "rotary":
        batch, seqlen, nheads, head_dim, half = (case[k] for k in ("batch", "seqlen", "nheads", "head_dim", "half"))
        x = torch.empty((batch, seqlen, nheads, head_dim), dtype=torch.float16, device="cuda").normal_(generator=gen)
        sin, cos = (torch.from_numpy(t).cuda() for t in synth.rotary_tables(seqlen, half))
        return {"op": "rotary", "x": x, "tables": (sin, cos), "args": (
            x.data_ptr(), sin.data_ptr(), cos.data_ptr(), batch, seqlen, nheads, head_dim, half,
            seqlen * nheads * head_dim, nheads * head_dim, head_dim)}
    T, N, state_len = case["T"], case["N"], case["state_len"]
    q_scale, q_shift = QUALITY[state_len]
    opt = api.DECODER_INIT(q_scale=q_scale, q_shift=q_shift)
    batches = []
    for _ in range(2 if case["op"] == "flight" else 1):
        x = _scores(case, gen)
        call = (T, N, case["columns"] * 4 ** state_len, x.data_ptr(), state_len, opt, api.GpuBuf(T, N, state_len))
        batches.append((x, call))
    return {"op": case["op"], "batches": batches}


def run(state):
    if state["op"] == "rotary":  # in place: the tensor is the result
        api.openfish_rotary_emb_gpu(*state["args"])
        return state["x"]
    calls = [call for _, call in state["batches"]]
    if state["op"] == "decode":
        return api.openfish_decode_gpu(*calls[0])
    for call in calls:
        api.openfish_amd_decode_enqueue(*call)
    return [api.openfish_amd_decode_wait(call[-1]) for call in calls]


def work(case):
    if case["op"] == "rotary":
        pairs = case["batch"] * case["seqlen"] * case["nheads"] * case["half"]
        return {"bytes": 2 * 4 * pairs + 2 * 4 * case["seqlen"] * case["half"], "flops": 6 * pairs}
    steps = case["T"] * case["N"] * (2 if case["op"] == "flight" else 1)
    S = 4 ** case["state_len"]
    # scores in; a byte of moves, bases and qualities out.  Per state and sweep: four additions, the maximum of
    # five, five differences, exponentials and additions, a logarithm and an addition; then the posterior
    return {"bytes": steps * (2 * case["columns"] * S + 3), "flops": steps * S * (2 * 25 + 5)}


def tolerance(case):
    if case["op"] == "rotary":
        return "exact"  # separate fp32 products and sums, rounded once
    # moves and bases are the CPU path's.  A quality character is a threshold on a quotient of posteriors, and the
    # sum below a posterior may be taken in any order: a sixth digit decides about 0.05 % of the characters
    return {"rel": 0.0, "differ": 5e-4}
