"""Every form of the rotary kernel (rotary.hip: rows, vec8, narrow with 4, 2 and 1 pairs) against the CPU path rounded to half, bit
for bit: at the sizes where the choice changes, odd batches, partly rotated heads, gaps between heads, transposed strides and
addresses that are not aligned for the wide loads.  What lies outside the rotated halves is untouched."""
import numpy as np
import pytest

from openfish_amd import synth
from oracle import crf_oracle as O
from test_gpu_parity import api  # noqa: F401

pytestmark = pytest.mark.gpu

# batch, seqlen, nheads, half: rows up to a half of 64, from 2048 lanes a batch (half / 4 lanes a head) and four batches up
SIZES = [(4, 1024, 1, 8), (4, 1023, 1, 8), (3, 1024, 1, 8), (5, 513, 1, 16), (4, 171, 3, 16), (5, 86, 3, 32), (7, 33, 4, 64), (4, 32, 4, 64), (4, 31, 4, 64), (4, 23, 3, 128),
         (5, 11, 3, 256), (4, 5, 4, 512), (3, 40, 3, 24), (3, 29, 3, 12), (2, 17, 5, 20), (3, 31, 2, 6), (2, 9, 3, 10), (3, 7, 5, 5), (1, 1, 1, 1)]


@pytest.mark.parametrize("layout", ["plain", "wide heads", "odd gap", "transposed", "address off by 2 bytes", "address off by 8 bytes"])
@pytest.mark.parametrize("batch,seqlen,nheads,half", SIZES)
def test_every_form_equals_the_cpu_path(api, batch, seqlen, nheads, half, layout):  # noqa: F811
    head = 2 * half + {"wide heads": 16, "odd gap": 3}.get(layout, 0)
    if layout == "transposed":  # heads outside, time steps inside
        strides = (nheads * seqlen * head, head, seqlen * head)
    else:
        strides = (seqlen * nheads * head, nheads * head, head)
    skip = {"address off by 2 bytes": 1, "address off by 8 bytes": 4}.get(layout, 0)
    n = batch * seqlen * nheads * head
    x16 = np.random.default_rng(n + skip).standard_normal(n + 8).astype(np.float16)
    sn, cs = synth.rotary_tables(seqlen, half)
    want = x16.copy()
    want[skip:skip + n] = O.rotary_emb(x16[skip:skip + n].astype(np.float32), sn, cs, batch, seqlen, nheads, head, half,
                                       *strides).reshape(-1).astype(np.float16)
    xd, sd, cd = (api.DeviceBuffer.from_host(v) for v in (x16, sn, cs))
    api.openfish_rotary_emb_gpu(xd.ptr + 2 * skip, sd, cd, batch, seqlen, nheads, head, half, *strides)
    assert np.array_equal(xd.to_host(np.float16, x16.shape).view(np.uint16), want.view(np.uint16))
