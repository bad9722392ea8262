"""The pinned memory behind a generation state's logits (llm_metal_amd/sft.py), with an allocator that only counts."""
import ctypes as C

import numpy as np

from llm_metal_amd.sft import _HostPool


class Counting:
    def __init__(self):
        self.live = {}

    def hip_host_alloc(self, n):
        b = C.create_string_buffer(n)
        self.live[C.addressof(b)] = b
        return C.addressof(b)

    def hip_host_free(self, p):
        del self.live[p]


def test_blocks_live_as_long_as_an_array_looks_at_them_and_are_bounded():
    lib = Counting()
    pool = _HostPool(lib)
    small = pool.empty((2, 8))
    assert not lib.live and small.shape == (2, 8)                    # ordinary memory
    a = pool.empty((3, 40000))
    a[:] = 2
    at, row = a.ctypes.data, a[1]
    del a
    assert not pool.idle and row.sum() == 80000                      # a view keeps its block
    del row
    b = pool.empty((3, 40000))
    assert b.ctypes.data == at and len(lib.live) == 1                # and the next array takes it
    pool.LIMIT = pool.held + 4 * 20000
    c, d = pool.empty((20000,)), pool.empty((20000,))
    assert len(lib.live) == 2 and d.dtype == np.float32              # d: beyond the limit, ordinary memory
    del c
    e = pool.empty((30000,))
    assert len(lib.live) == 1                                        # no room beside b, idle blocks were given up for it
    pool.close()
    assert len(lib.live) == 1
    b += 1                                                           # an array outlives the state
    del b
    assert not lib.live and pool.held == 0
    assert pool.empty((40000,)).size == 40000 and not lib.live
    del d, e
