"""A decode's results are arrays over what the C API returned by malloc: each buffer is freed once, with the last array over it."""
import ctypes as C
import gc

import numpy as np

from openfish_amd import api


def test_a_taken_buffer_lives_as_long_as_an_array_over_it(monkeypatch):
    freed = []
    monkeypatch.setattr(api._Malloced.__init__, "__defaults__", (freed.append,))
    store = (C.c_uint8 * 6)(*range(6))
    address = C.addressof(store)
    a = api._take(C.c_void_p(address), 2, 3)
    assert a.shape == (2, 3) and a.dtype == np.uint8 and a.flags.c_contiguous and a.flags.writeable
    assert np.array_equal(a, [[0, 1, 2], [3, 4, 5]])
    row = a[1]
    row[0] = 9
    assert store[3] == 9
    del a
    gc.collect()
    assert freed == [] and row.tolist() == [9, 4, 5]
    del row
    gc.collect()
    assert freed == [address]
