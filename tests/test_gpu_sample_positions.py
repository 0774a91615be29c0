"""The sampled boundaries of the partition forms: data with a period that
divides the sample's stride is sampled from every phase, and inputs built on
the sampled positions themselves still take the paths for buckets that the
sample missed."""
import numpy
import pytest

from gpu_util import even
from mpsort import _lib, segments, workloads
from mpsort._lib import lib
from test_gpu_direct import note, ragged
from test_gpu_histsort import check_parity
from test_gpu_segments import expected, make

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def no_options():
    lib.mpsort_mpi_unset_options(-1)


def positions(m, n):
    """sample_pos of lsort_dev.h for u = 0 .. m - 1"""
    u = numpy.arange(m, dtype=numpy.uint64)
    h = u.copy()
    for shift, mul in ((16, 0x85ebca6b), (13, 0xc2b2ae35), (16, 1)):
        h = ((h ^ (h >> numpy.uint64(shift))) * numpy.uint64(mul)) & numpy.uint64(0xffffffff)
    return ((((u << numpy.uint64(16)) | (h & numpy.uint64(0xffff))) * numpy.uint64(n)) >> numpy.uint64(16)) // numpy.uint64(m)


def test_positions_cover_the_records():
    for m, n in ((1024, 8193), (4096, 4096), (4096, 100003), (16384, (1 << 29) - 1)):
        p = positions(m, n).astype(numpy.int64)
        u = numpy.arange(m)
        assert (p >= u * n // m).all() and (p <= ((u + 1) * n - 1) // m).all() and p[-1] < n


def interleaved(n, period, seed):
    """records of period sources in turn, each source with keys of its own"""
    k = numpy.random.default_rng(seed).integers(0, 1 << 40, n, dtype=numpy.uint64)
    return k | ((numpy.arange(n, dtype=numpy.uint64) % numpy.uint64(period)) << numpy.uint64(40))


# (records, sources): the sample's stride is the number of sources
@pytest.mark.parametrize("n, period, form", [(1 << 21, 128, _lib.FORM_ONE_LEVEL), (1 << 23, 4096, _lib.FORM_TWO_LEVELS),
                                             (1 << 23, 64, _lib.FORM_TWO_LEVELS)])
@pytest.mark.parametrize("P", [1, 8])
def test_interleaved_sources(n, period, form, P):
    note("interleaved n=%d period=%d P=%d" % (n, period, P))
    out, st = check_parity(workloads.records16(interleaved(n, period, 1)), even(n, P), even(n, P), 'key', device=True)
    assert st.form == form
    assert st.buckets_overflow == 0 and st.buckets_listed * 20 < st.buckets


def test_interleaved_segments_take_no_longer():
    """a batched segment of 2^19 records of 128 interleaved sources against one
    of the same keys in random order"""
    n = 1 << 19
    k = interleaved(n, 128, 2)
    d, o = lib.mpsort_gpu_dmalloc(16 * n), lib.mpsort_gpu_dmalloc(16 * n)
    ms = []
    try:
        for keys in (numpy.random.default_rng(3).permutation(k), k):
            a = numpy.zeros(n, workloads.REC16I)
            a['key'], a['value'] = keys.astype(numpy.int64), numpy.arange(n)
            _lib.check(lib.mpsort_gpu_memcpy_h2d(d, a.ctypes.data, a.nbytes))
            plan = segments.SegmentPlan()
            plan.add(d, o, [n], a.dtype, 'key')
            ms.append(min(plan.run() for _ in range(5)))
            g = numpy.empty_like(a)
            _lib.check(lib.mpsort_gpu_memcpy_d2h(g.ctypes.data, o, a.nbytes))
            plan.close()
            assert numpy.array_equal(g, expected(a, [n]))
    finally:
        lib.mpsort_gpu_dfree(d)
        lib.mpsort_gpu_dfree(o)
    note("random order %.3f ms, interleaved %.3f ms" % tuple(ms))
    assert ms[1] < 2 * ms[0]


def test_oversized_bucket_of_one_level():
    """every sampled position of one key: the keys above it share one bucket,
    which the radix path sorts"""
    n, P, S = 1 << 20, 5, 8192
    k = numpy.random.default_rng(3).integers(10, 1 << 62, n, dtype=numpy.uint64)
    k[positions(S, n).astype(numpy.int64)] = 5
    out, st = check_parity(workloads.records16(k), ragged(n, P, 9), ragged(n, P, 10), 'key', device=True)
    assert st.form == _lib.FORM_ONE_LEVEL and st.buckets_overflow == 1


@pytest.mark.parametrize("rec", ["rec16", "rows24"])
def test_coarse_bucket_beyond_the_runs(rec):
    """every sampled position of one key, so that all others share a coarse
    bucket of more tiles than a fine bucket gathers from: the call takes the
    per-rank form"""
    n, P, S = 6397953, 2, 2048
    k = numpy.random.default_rng(3).integers(1 << 20, 1 << 62, n).astype(numpy.uint64)
    k[positions(S, n).astype(numpy.int64)] = 5
    a = workloads.records16(k)
    if rec == "rows24":
        a = numpy.zeros(n, [('v', 'i8', 2), ('key', 'u8')])
        a['key'], a['v'] = k, numpy.arange(2 * n).reshape(n, 2)
    out, st = check_parity(a, ragged(n, P, 9), ragged(n, P, 10), 'key', device=True)
    assert st.form == _lib.FORM_RANKS


@pytest.mark.parametrize("dtype", [workloads.REC8, workloads.REC16I], ids=["8B", "16B"])
def test_segments_whose_sample_misses_the_weight(dtype):
    """every sampled position of one key: the other keys share a bucket above
    the in-LDS capacity, replayed on new contents, with eager work between
    the replays"""
    sizes = numpy.array([100003, 700, 60001], numpy.int64)
    nb = int(sizes.sum()) * dtype.itemsize
    d, o = lib.mpsort_gpu_dmalloc(nb), lib.mpsort_gpu_dmalloc(nb)
    plan = segments.SegmentPlan(graph=True)
    try:
        for rep in range(4):
            a = make(dtype, sizes, 31 + rep)
            b = 0
            for n in sizes if rep != 2 else ():
                if n > 4096:
                    a['key'][b + positions(4096, n).astype(numpy.int64)] = -7
                b += n
            _lib.check(lib.mpsort_gpu_memcpy_h2d(d, a.ctypes.data, a.nbytes))
            if rep == 0:
                plan.add(d, o, sizes, a.dtype, 'key')
            plan.run()
            g = numpy.empty_like(a)
            _lib.check(lib.mpsort_gpu_memcpy_d2h(g.ctypes.data, o, a.nbytes))
            assert numpy.array_equal(g, expected(a, sizes)), rep
            small = make(dtype, [5000], 3)
            assert numpy.array_equal(segments.sort_segments(small, [5000], 'key'), expected(small, [5000]))
    finally:
        plan.close()
        lib.mpsort_gpu_dfree(d)
        lib.mpsort_gpu_dfree(o)
