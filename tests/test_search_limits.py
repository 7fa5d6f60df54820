"""What the launchers of the beam search refuse before anything is queued: chunks longer than the maps of the traceback, which lie in LDS,
have room for.  The library's entry points refuse them as well; this is the launchers' own check, so no device is needed."""
import ctypes as C

import pytest

from openfish_amd import api

MAX_T, BAD_ARGS = 8192, -1
AT = C.c_void_p(4096)  # any aligned address: nothing reads it


def search(T, state_len, columns, entry):
    shape = [C.c_int(T), C.c_int(1), C.c_int(state_len), C.c_int(columns), C.c_float(2.0), C.c_float(2.0)]
    if entry == "static":
        return api.lib().ofk_beam_search_static(*[AT] * 4, *shape, C.c_int(0), C.c_void_p())
    if entry == "forward":
        return api.lib().ofk_beam_search_forward(*[AT] * 6, *shape, AT, C.c_int(0), C.c_void_p(), C.c_void_p())
    return api.lib().ofk_beam_search(*[AT] * 5, *shape, AT, C.c_int(0), C.c_void_p(), C.c_void_p())


@pytest.mark.parametrize("T", [MAX_T + 1, 2 ** 31 - 1])
@pytest.mark.parametrize("columns", [4, 5])
@pytest.mark.parametrize("state_len,entry", [(3, "plain"), (4, "plain"), (5, "plain"), (4, "forward"), (5, "forward"), (3, "static"), (5, "static")])
def test_longer_chunks_are_refused(T, columns, state_len, entry):
    assert search(T, state_len, columns, entry) == BAD_ARGS
