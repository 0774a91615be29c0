"""Device allocations that fail, through the allocator hook: a call that the
per-rank form has memory for still succeeds, and a failed call leaves the
caller's output as it was."""
import ctypes

import numpy
import pytest

from gpu_util import even, key_desc
from mpsort import _lib
from mpsort._lib import lib
from test_gpu_direct import note
from test_gpu_sample_positions import positions

pytestmark = pytest.mark.gpu

MALLOC = ctypes.CFUNCTYPE(ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p)
FREE = ctypes.CFUNCTYPE(None, ctypes.c_void_p, ctypes.c_void_p)


class Allocator(object):
    """the library's device allocations, of which fails(index, bytes, held) do"""

    def __init__(self, fails):
        self.fails, self.sizes, self.count, self.failed = fails, {}, 0, 0
        self.m, self.f = MALLOC(self._malloc), FREE(self._free)

    def _malloc(self, nbytes, _):
        self.count += 1
        if self.fails(self.count - 1, nbytes, sum(self.sizes.values())):
            self.failed += 1
            return None
        p = lib.mpsort_gpu_dmalloc(nbytes)
        self.sizes[p] = nbytes
        return p

    def _free(self, p, _):
        del self.sizes[p]
        lib.mpsort_gpu_dfree(p)

    def __enter__(self):
        lib.mpsort_gpu_set_allocator(self.m, self.f, None)
        return self

    def __exit__(self, *a):
        lib.mpsort_gpu_set_allocator(MALLOC(), FREE(), None)  # frees all that the hook gave
        assert not self.sizes


@pytest.fixture(autouse=True)
def no_options():
    lib.mpsort_mpi_unset_options(-1)


def sort_into_marked(a, P, field='key', flags=0):
    """(return code, output) of a device sort into memory filled with 0x5a"""
    d, o = lib.mpsort_gpu_dmalloc(a.nbytes), lib.mpsort_gpu_dmalloc(a.nbytes)
    try:
        out = numpy.full(a.nbytes, 0x5a, numpy.uint8)
        _lib.check(lib.mpsort_gpu_memcpy_h2d(d, a.ctypes.data, a.nbytes))
        _lib.check(lib.mpsort_gpu_memcpy_h2d(o, out.ctypes.data, a.nbytes))
        c = (ctypes.c_int64 * P)(*even(len(a), P))
        k = key_desc(a.dtype, field)
        rc = lib.mpsort_gpu_newarray(d, c, P, o, c, a.dtype.itemsize, ctypes.byref(k), flags | _lib.DEVICE_PTRS)
        _lib.check(lib.mpsort_gpu_memcpy_d2h(out.ctypes.data, o, a.nbytes))
    finally:
        lib.mpsort_gpu_dfree(d)
        lib.mpsort_gpu_dfree(o)
    return rc, out


@pytest.mark.parametrize("itemsize", [24, 32])
def test_failed_call_leaves_the_output(itemsize):
    """packed records whose coarse buckets the sample misses: the two-level
    sort gives the call up for the per-rank form, and each allocation of the
    two fails in turn"""
    n, P = 6397953, 2
    dt = numpy.dtype({"names": ["key", "v"], "formats": ["<u8", "<i8"], "offsets": [8, 16], "itemsize": itemsize})
    a = numpy.zeros(n, dt)
    a['key'] = numpy.random.default_rng(3).integers(1 << 20, 1 << 62, n)
    a['key'][positions(2048, n).astype(numpy.int64)] = 5
    a['v'] = numpy.arange(n)
    want = a[numpy.argsort(a['key'], kind='stable')].view(numpy.uint8)
    fail = 0
    while True:
        with Allocator(lambda i, nbytes, held: i == fail) as al:
            rc, out = sort_into_marked(a, P)
        note("allocation %d of %d fails: rc %d" % (fail, al.count, rc))
        if rc:
            assert rc == _lib.MPSORT_ERR_NOMEM
            assert (out == 0x5a).all()
        else:
            assert numpy.array_equal(out, want)
        if not al.failed:
            break
        fail += 1
    assert fail > 4


@pytest.mark.parametrize("rec, n, P, first", [("rec16", 5000011, 1, _lib.FIRST_RADIX),
                                              ("rows24", 5000011, 4, _lib.FIRST_BUCKETS)])
def test_memory_of_the_per_rank_form_suffices(rec, n, P, first):
    """device memory for what the per-rank form holds (first: the FirstSort
    it takes at this size), but not for the two-level form's buffers"""
    g = numpy.random.default_rng(n)
    a = numpy.zeros(n, [('key', 'u8'), ('v', 'i8')] if rec == "rec16" else [('v', 'i8', 2), ('key', 'u8')])
    a['key'] = g.integers(0, 1 << 40, n)
    a['v'] = numpy.arange(a['v'].size).reshape(a['v'].shape)
    want = a[numpy.argsort(a['key'], kind='stable')].view(numpy.uint8)
    with Allocator(lambda i, nbytes, held: False) as al:
        rc, out = sort_into_marked(a, P, flags=first)
        assert rc == 0 and lib.mpsort_gpu_last_form() == _lib.FORM_RANKS
        budget = sum(al.sizes.values())
    with Allocator(lambda i, nbytes, held: held + nbytes > budget) as al:
        rc, out = sort_into_marked(a, P)
        note("n=%d: %d bytes held, budget %d, %d allocations failed" % (n, sum(al.sizes.values()), budget, al.failed))
        assert rc == 0, lib.mpsort_gpu_last_error()
        assert al.failed and lib.mpsort_gpu_last_form() == _lib.FORM_RANKS
        assert numpy.array_equal(out, want)
        rc, out = sort_into_marked(a, P)  # and again, with what the first call left allocated
        assert rc == 0 and numpy.array_equal(out, want)
