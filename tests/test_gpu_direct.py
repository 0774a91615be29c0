"""The sort of up to 64 ranks without per-rank local sorts: one partition over
all ranks, in-LDS bucket sorts, the counts read off the result.  Held to the
oracle's bytes and counts at the edges of its sizes (one tile, one bucket more,
the largest single partition), of ranks and tiles, and on keys that strain the
sampled boundaries."""
import sys

import numpy
import pytest

from gpu_util import even
from mpsort import _lib, workloads
from mpsort._lib import lib
from test_gpu_histsort import check_parity
from test_gpu_plain_merged import keys

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def no_options():
    lib.mpsort_mpi_unset_options(-1)


def note(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def ragged(n, P, seed):
    cut = numpy.sort(numpy.random.default_rng(seed).integers(0, n + 1, P - 1))
    return numpy.diff(numpy.concatenate([[0], cut, [n]]))


@pytest.mark.parametrize("n", [8193, 3072 * 3, 2 * 8192, 2048 * 16 + 1, 2048 * 512 + 1, 2048 * 1024 + 1, 4300800, 4300801])
def test_sizes(n):
    P = 5
    a = workloads.records16(keys("random", n, n % 97))
    note("direct n=%d" % n)
    check_parity(a, ragged(n, P, 1), ragged(n, P, 2), 'key', device=True)


@pytest.mark.parametrize("shape", ["heavy", "few", "zero_heavy", "sorted", "reversed", "narrow", "two_scales"])
@pytest.mark.parametrize("P", [1, 63, 64])
def test_shapes(shape, P):
    n = 300007
    a = workloads.records16(keys(shape, n, 5 + P))
    note("direct shape=%s P=%d" % (shape, P))
    check_parity(a, ragged(n, P, 3), ragged(n, P, 4), 'key', device=True)


@pytest.mark.parametrize("P", [2, 64])
@pytest.mark.parametrize("value", [0, 1, 2 ** 64 - 1])
def test_one_key_value(value, P):
    """every record one key, the smallest and the largest value among them;
    and one other key in front of, or behind, the heavy one"""
    n = 50021
    k = numpy.full(n, value, numpy.uint64)
    check_parity(workloads.records16(k), ragged(n, P, 5), ragged(n, P, 6), 'key', device=True)
    k[n // 2] = numpy.uint64(value - 1 if value > 1 else value + 1)
    check_parity(workloads.records16(k), ragged(n, P, 5), ragged(n, P, 6), 'key', device=True)


@pytest.mark.parametrize("dt", ["u8", "i8", "i4pair", "u4pair", "keytail"])
def test_record_types(dt):
    n, P = 61001, 9
    g = numpy.random.default_rng(8)
    if dt in ("u8", "i8"):
        i = numpy.iinfo(dt)
        a, f = g.integers(i.min, i.max, n, dtype=dt, endpoint=True), None
    elif dt == "keytail":
        a, f = numpy.zeros(n, [('v', 'i8'), ('key', 'i8')]), 'key'
        a['key'], a['v'] = g.integers(-300, 300, n), numpy.arange(n)
    else:
        a, f = numpy.zeros(n, [('key', dt[:2]), ('v', 'f4')]), 'key'
        i = numpy.iinfo(dt[:2])
        a['key'], a['v'] = g.integers(i.min, i.max, n, dtype=dt[:2], endpoint=True), numpy.arange(n)
    check_parity(a, ragged(n, P, 7), ragged(n, P, 8), f, device=True)


def test_overlapping_output():
    """input and output overlap without being equal: the input is read whole
    before the output is written"""
    import ctypes
    from gpu_util import key_desc
    n, P, shift = 70001, 3, 1024
    a = workloads.records16(keys("heavy", n, 3))
    want = a[numpy.argsort(a['key'], kind='stable')]
    d = lib.mpsort_gpu_dmalloc((n + shift) * 16)
    try:
        _lib.check(lib.mpsort_gpu_memcpy_h2d(d, a.ctypes.data, a.nbytes))
        c = (ctypes.c_int64 * P)(*even(n, P))
        k = key_desc(a.dtype, 'key')
        _lib.check(lib.mpsort_gpu_newarray(d, c, P, d + shift * 16, c, 16, ctypes.byref(k), _lib.DEVICE_PTRS))
        out = numpy.empty_like(a)
        _lib.check(lib.mpsort_gpu_memcpy_d2h(out.ctypes.data, d + shift * 16, a.nbytes))
    finally:
        lib.mpsort_gpu_dfree(d)
    assert numpy.array_equal(out, want)


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 1023, 1024, 1025, 4095, 4096, 4097, 8191, 8192])
@pytest.mark.parametrize("P", [1, 2, 64])
def test_one_workgroup_sizes(n, P):
    a = workloads.records16(keys("random", n, n))
    out, st = check_parity(a, ragged(n, P, 9), ragged(n, P, 10), 'key', device=True)
    assert st.first_passes <= 8


@pytest.mark.parametrize("shape", ["heavy", "few", "zero_heavy", "sorted", "narrow", "two_scales"])
def test_one_workgroup_shapes(shape):
    P = 17
    for n in (3001, 5003):
        check_parity(workloads.records16(keys(shape, n, 12)), ragged(n, P, 11), ragged(n, P, 12), 'key')


@pytest.mark.parametrize("dt", ["u4", "i4", "u8", "i8", "particle32", "rec24", "rec13", "keytail"])
@pytest.mark.parametrize("n, inplace", [(2003, False), (2003, True), (6007, False), (6007, True)])
def test_one_workgroup_record_types(dt, n, inplace):
    """4-, 8-, 16- and 32-byte records directly, others (24 bytes; 13 bytes
    with a key at an odd offset) from their bytes; in place too"""
    import oracle
    from gpu_util import gpu_sort_device, last_counts
    from test_gpu_histsort import _device_inplace
    P = 6
    g = numpy.random.default_rng(14)
    if dt in ("u4", "i4", "u8", "i8"):
        i = numpy.iinfo(dt)
        a, f = g.integers(i.min, i.max, n, dtype=dt, endpoint=True), None
    else:
        t = {"particle32": workloads.PARTICLE32, "rec24": [('x', 'f8'), ('id', 'i8'), ('w', 'u8')],
             "rec13": [('b', 'u1'), ('id', 'i4'), ('w', 'u8')], "keytail": [('v', 'i8'), ('id', 'i8')]}[dt]
        a, f = numpy.zeros(n, t), 'id'
        a.view(numpy.uint8).reshape(n, -1)[:] = g.integers(0, 256, (n, a.dtype.itemsize))
        a['id'] = g.integers(0, 900, n)
    note("one workgroup %s n=%d inplace=%s" % (dt, n, inplace))
    ref, info = oracle.histogram_sort(a, even(n, P), even(n, P), oracle.key_for(a.dtype, f))
    out, st = _device_inplace(a, even(n, P), f) if inplace else gpu_sort_device(a, even(n, P), even(n, P), f)
    assert numpy.array_equal(out.view(numpy.uint8), ref.view(numpy.uint8))
    c = last_counts(P, 8)
    for k in ("P", "C", "myCLT", "myCLE", "myC", "send"):
        assert numpy.array_equal(c[k], info[k]), k
    assert st.checksum_in == info['checksum_in'] == st.checksum_out


@pytest.mark.parametrize("n", [8193, 262145, 2048 * 1024 - 1, 2048 * 1024 + 1])
@pytest.mark.parametrize("at", [0, 12, 24])
def test_packed_32_byte_records(n, at):
    """32-byte records sorted as packed {key, index}: the pack and the gather
    at the edges of their blocks and of one round of them, with the key at
    several places"""
    dt = numpy.dtype({"names": ["key", "a", "b"], "formats": ["<i8", "<u4", "<u4"],
                      "offsets": [at, (at + 8) % 32, (at + 16) % 32], "itemsize": 32})
    g = numpy.random.default_rng(n + at)
    a = numpy.frombuffer(g.bytes(32 * n), dt).copy()
    a['key'] >>= 30
    P = 7
    check_parity(a, ragged(n, P, 1), ragged(n, P, 2), 'key', flags=_lib.FORCE_GENERAL, device=True)
