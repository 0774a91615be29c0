"""Records of one key sorted in place in device memory: no digit pass runs, and
the output's checksum is still taken."""
import ctypes

import numpy
import pytest

from gpu_util import even, key_desc
from mpsort import _lib, workloads
from mpsort._lib import lib
from test_gpu_direct import note

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def no_options():
    lib.mpsort_mpi_unset_options(-1)


@pytest.mark.parametrize("entry", ["newarray", "newarray_noalloc"])
@pytest.mark.parametrize("flags", [0, _lib.FIRST_RADIX, _lib.FIRST_BUCKETS], ids=["default", "radix", "buckets"])
@pytest.mark.parametrize("rec", ["u4", "u8", "rec16", "wide_key", "particle32", "rows24"])
@pytest.mark.parametrize("n, P", [(5, 1), (7001, 1), (30011, 1), (30011, 3)])
def test_one_key_in_place(rec, n, P, flags, entry):
    g = numpy.random.default_rng(n)
    field = None
    if rec in ("u4", "u8"):
        a = numpy.full(n, 0x01020384, rec)
    else:
        t, field = {"rec16": ([('key', 'u8'), ('v', 'i8')], 'key'), "wide_key": ([('key', 'u8', 2)], 'key'),
                    "particle32": (workloads.PARTICLE32, 'id'), "rows24": ([('v', 'i8', 2), ('key', 'u8')], 'key')}[rec]
        a = numpy.frombuffer(g.bytes(n * numpy.dtype(t).itemsize), t).copy()
        a[field] = 0x01020384
    note("one key in place %s n=%d P=%d flags=%d %s" % (rec, n, P, flags, entry))
    d = lib.mpsort_gpu_dmalloc(a.nbytes)
    try:
        _lib.check(lib.mpsort_gpu_memcpy_h2d(d, a.ctypes.data, a.nbytes))
        c = (ctypes.c_int64 * P)(*even(n, P))
        k = key_desc(a.dtype, field)
        _lib.check(getattr(lib, "mpsort_gpu_" + entry)(d, c, P, d, c, a.dtype.itemsize, ctypes.byref(k),
                                                       flags | _lib.DEVICE_PTRS))
        out = numpy.empty_like(a)
        _lib.check(lib.mpsort_gpu_memcpy_d2h(out.ctypes.data, d, a.nbytes))
    finally:
        lib.mpsort_gpu_dfree(d)
    st = _lib.last_stats()
    assert numpy.array_equal(out.view(numpy.uint8), a.view(numpy.uint8))
    assert st.checksum_in == st.checksum_out == int(a.view(numpy.int8).sum(dtype=numpy.int64))
