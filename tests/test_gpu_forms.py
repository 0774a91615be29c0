"""Which form sorts a call's records (mpsort_gpu_last_form): by size and record
type, and the reference's per-rank steps with the merged SecondSort where the
FirstSort's form is asked for, on the inputs that strain it.  Every result
is held to the oracle's bytes and counts."""
import ctypes
import sys

import numpy
import pytest

from gpu_util import even, gpu_sort, gpu_sort_device
from mpsort import _lib, learned, workloads
from mpsort._lib import lib
from test_gpu_direct import ragged
from test_gpu_histsort import check_parity
from test_gpu_learned import keys_of, trained
from test_gpu_plain_merged import SHAPES, keys

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def no_options():
    lib.mpsort_mpi_unset_options(-1)


def note(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("n, form", [(1, _lib.FORM_ONE_LAUNCH), (8192, _lib.FORM_ONE_LAUNCH), (8193, _lib.FORM_ONE_LEVEL),
                                     (4300800, _lib.FORM_ONE_LEVEL), (4300801, _lib.FORM_TWO_LEVELS)])
def test_form_by_size(n, form):
    a = workloads.records16(keys("random", n, 3))
    out, st = check_parity(a, ragged(n, 5, 1), ragged(n, 5, 2), 'key', device=True)
    assert st.form == form
    assert st.bisect_rounds == 0 and st.first_passes <= 8 and st.second_passes == 0


@pytest.mark.parametrize("past, form", [(0, _lib.FORM_TWO_LEVELS), (1, _lib.FORM_RANKS)])
def test_the_largest_two_level_sort(past, form):
    """sorted, and the same keys: as many of every top 16 bits, and equal sums
    and exclusive ors"""
    n, P = 512 * 256 * 6144 // 16 * 7 + past, 3
    note("two levels at their largest, n=%d" % n)
    a = numpy.random.default_rng(5).integers(0, 2 ** 64, n, dtype=numpy.uint64)
    out, st = gpu_sort_device(a, ragged(n, P, 1), ragged(n, P, 2))
    assert st.form == form
    assert (out[1:] >= out[:-1]).all()
    top = lambda x: numpy.bincount((x >> numpy.uint64(48)).astype(numpy.uint16), minlength=1 << 16)
    assert numpy.array_equal(top(out), top(a))
    assert out.sum() == a.sum() and numpy.bitwise_xor.reduce(out) == numpy.bitwise_xor.reduce(a)


@pytest.mark.parametrize("P, itemsize, n, form", [
    (5, 1024, 4096, _lib.FORM_ONE_LAUNCH), (5, 1024, 4097, _lib.FORM_RANKS), (5, 1024, 8192, _lib.FORM_RANKS),
    (5, 256, 8192, _lib.FORM_ONE_LAUNCH), (5, 260, 8192, _lib.FORM_RANKS), (5, 128, 8192, _lib.FORM_ONE_LAUNCH),
    (5, 127, 8192, _lib.FORM_ONE_LAUNCH), (5, 129, 8192, _lib.FORM_RANKS), (5, 1023, 4096, _lib.FORM_ONE_LAUNCH),
    (5, 1023, 4097, _lib.FORM_RANKS), (5, 65536, 17, _lib.FORM_ONE_LAUNCH),
    (1, 64, 8192, _lib.FORM_ONE_LAUNCH), (1, 68, 8192, _lib.FORM_RANKS), (1, 31, 8192, _lib.FORM_ONE_LAUNCH),
    (1, 33, 8192, _lib.FORM_RANKS), (1, 1023, 4096, _lib.FORM_ONE_LAUNCH)])
def test_form_of_wide_records(P, itemsize, n, form):
    """records of more bytes than one workgroup should move are spread over
    the chip: both sides of 4096 records and of the bounds in
    bytes"""
    dt = numpy.dtype({"names": ["key"], "formats": ["<u8"], "offsets": [itemsize // 2], "itemsize": itemsize})
    g = numpy.random.default_rng(itemsize)
    a = numpy.frombuffer(g.bytes(itemsize * n), dt).copy()
    a['key'] >>= 52
    out, st = check_parity(a, ragged(n, P, 1), ragged(n, P, 2), 'key', device=True)
    assert st.form == form


@pytest.mark.parametrize("inplace", [False, True])
@pytest.mark.parametrize("itemsize", [8, 16])
@pytest.mark.parametrize("P", [1, 64])
def test_one_key_takes_no_longer(itemsize, P, inplace):
    """4,000,000 records of one key, checksum included, against random keys;
    in place they take the path of oversized buckets"""
    n = 4000000
    c = (ctypes.c_int64 * P)(*even(n, P))
    key = _lib.KeyDesc(offset=0, width=8, is_signed=0, nwords=1, reserved=0)
    d = lib.mpsort_gpu_dmalloc(n * itemsize)
    o = d if inplace else lib.mpsort_gpu_dmalloc(n * itemsize)
    ms = []
    try:
        for k in (keys("random", n, 1), numpy.full(n, 77, numpy.uint64)):
            a = numpy.zeros((n, itemsize // 8), numpy.uint64)
            a[:, -1] = numpy.arange(n)
            a[:, 0] = k
            t = []
            for _ in range(5):
                _lib.check(lib.mpsort_gpu_memcpy_h2d(d, a.ctypes.data, a.nbytes))
                _lib.check(lib.mpsort_gpu_newarray(d, c, P, o, c, itemsize, ctypes.byref(key), _lib.DEVICE_PTRS))
                t.append(_lib.last_stats().t_total_ms)
            ms.append(min(t))
            assert _lib.last_stats().form == _lib.FORM_ONE_LEVEL
            out = numpy.empty_like(a)
            _lib.check(lib.mpsort_gpu_memcpy_d2h(out.ctypes.data, o, a.nbytes))
            assert numpy.array_equal(out, a[numpy.argsort(a[:, 0], kind='stable')])
    finally:
        lib.mpsort_gpu_dfree(d)
        if not inplace:
            lib.mpsort_gpu_dfree(o)
    note("random keys %.3f ms, one key %.3f ms" % tuple(ms))
    assert ms[1] < (4 if inplace else 2) * ms[0]


@pytest.mark.parametrize("why", ["ranks", "wide key", "4-byte records", "exchange", "radix FirstSort", "bucket FirstSort"])
def test_calls_that_keep_the_ranks(why):
    n, P, flags, field = 30000, 65 if why == "ranks" else 4, 0, 'key'
    a = workloads.records16(keys("heavy", n, 3))
    if why == "wide key":
        a = numpy.zeros(n, [('key', 'u8', 2)])
        a['key'] = numpy.random.default_rng(1).integers(0, 99, (n, 2))
    elif why == "4-byte records":
        a, field = numpy.random.default_rng(1).integers(0, 999, n, dtype=numpy.uint32), None
    else:
        flags = {"exchange": _lib.EXCHANGE, "radix FirstSort": _lib.FIRST_RADIX,
                 "bucket FirstSort": _lib.FIRST_BUCKETS}.get(why, 0)
    out, st = check_parity(a, even(n, P), even(n, P), field, flags=flags, device=True)
    assert st.form == _lib.FORM_RANKS


@pytest.mark.parametrize("n, form", [(200000, _lib.FORM_RANKS), (4300801, _lib.FORM_TWO_LEVELS)])
def test_learned_form(n, form):
    P = 16
    model = trained("uniform", n)
    try:
        a = workloads.records16(keys_of("uniform", n, 5))
        ref, _ = gpu_sort(a, even(n, P), even(n, P), 'key')
        out = learned.sort_learned(a, model, 'key', nin=even(n, P))
        st = _lib.last_stats()
    finally:
        model.close()
    assert numpy.array_equal(out, ref)
    assert st.form == form and st.learned == 1
    assert st.splitters_exact + st.splitters_repaired == P - 1
    assert (st.repair_rounds == 0) == (form == _lib.FORM_TWO_LEVELS)


def test_no_form_after_a_failed_or_empty_call():
    a = workloads.records16(keys("random", 10, 1))
    gpu_sort(a, [10], [10], 'key')
    assert _lib.last_stats().form == _lib.FORM_ONE_LAUNCH
    with pytest.raises(ValueError):
        gpu_sort(a, [10], [9], 'key')
    assert lib.mpsort_gpu_last_form() == _lib.FORM_NONE
    gpu_sort(a, [10], [10], 'key')
    out, st = gpu_sort(a[:0], [0], [0], 'key')
    assert st.form == _lib.FORM_NONE


# The merged SecondSort after either FirstSort: calls that ask for one are
# sorted rank by rank, whatever their size.

FIRST = pytest.mark.parametrize("first", [_lib.FIRST_RADIX, _lib.FIRST_BUCKETS], ids=["radix", "buckets"])


def merged(a, nin, nout, field, flags):
    out, st = check_parity(a, nin, nout, field, flags=flags, device=True)
    assert st.form == _lib.FORM_RANKS and st.second_merged == 1
    assert st.exchange_runs == 0 and st.second_passes == 0 and st.plain_sides == 0
    return st


@FIRST
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("P", [2, 5, 64])
def test_merged_second_sort_shapes(shape, P, first):
    n = 60000 + 101 * P
    note("merged after FirstSort flags=%d shape=%s P=%d" % (first, shape, P))
    merged(workloads.records16(keys(shape, n, 7 + P)), even(n, P), even(n, P), 'key', first)


@FIRST
@pytest.mark.parametrize("P", [3, 64])
def test_merged_ragged_and_empty_receivers(P, first):
    n = 40000
    a = workloads.records16(keys("random", n, P))
    nout = numpy.zeros(P, numpy.int64)
    nout[0], nout[-1] = n // 3, n - n // 3  # every rank between receives nothing
    merged(a, ragged(n, P, P), nout, 'key', first)


@FIRST
def test_merged_large_receivers(first):
    """receivers of 65536 records, more than the 12288 samples of their tables"""
    n, P = 1 << 22, 64
    merged(workloads.clustered_records(n, seed=4), even(n, P), even(n, P), 'key', first)


@FIRST
@pytest.mark.parametrize("kind", ["u8", "i8", "u4_pairs", "rows24"])
def test_merged_record_types(kind, first):
    n, P = 50000, 16
    g = numpy.random.default_rng(11)
    if kind in ("u8", "i8"):
        i = numpy.iinfo(kind)
        a, field = g.integers(i.min, i.max, n, dtype=kind, endpoint=True), None
    else:
        t = [('key', 'u4'), ('v', 'u4')] if kind == "u4_pairs" else [('v', 'f8'), ('key', 'i8'), ('w', 'u8')]
        a, field = numpy.zeros(n, t), 'key'
        a['key'], a['v'] = g.integers(0, 1000, n), numpy.arange(n)
    st = merged(a, even(n, P), even(n, P), field, first)
    assert st.general_path == (kind == "rows24")


def test_merged_32_byte_records_are_packed():
    """ranks of 2^18 32-byte records after the bucket FirstSort"""
    n, P = 1 << 20, 4
    a = numpy.zeros(n, workloads.PARTICLE32)
    g = numpy.random.default_rng(21)
    a['id'] = g.permutation(n)
    a['id'][g.random(n) < 0.01] = 7
    a['pos'] = g.random((n, 3))
    st = merged(a, even(n, P), even(n, P), 'id', _lib.FIRST_BUCKETS)
    assert st.general_path == 1 and st.first_passes == 0
