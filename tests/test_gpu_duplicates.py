"""Keys that repeat: in-LDS sorts whose bins hold one key value many times
(placed by counting, 64 such bins at a time) or a heavy key among others, in
every workgroup shape, and what they cost next to distinct keys."""
import numpy
import pytest

from mpsort import _lib, segments, workloads
from mpsort._lib import lib
from test_gpu_direct import note, ragged
from test_gpu_histsort import check_parity
from test_gpu_segments import expected, _plan_sort

pytestmark = pytest.mark.gpu

# around the capacities of the workgroup shapes
SIZES = [9216, 9000, 4609, 4608, 4600, 3072, 3000, 1537, 1536, 1500, 769, 768, 700, 129, 128, 65]


@pytest.fixture(autouse=True)
def no_options():
    lib.mpsort_mpi_unset_options(-1)


def repeated(n, times, seed):
    """n keys, each value about `times` times, values spread out"""
    g = numpy.random.default_rng(seed)
    return (g.permutation(n) // times).astype(numpy.int64)


def records(dtype, keys, stretch):
    a = numpy.zeros(len(keys), dtype)
    a['key'] = (keys * stretch) if dtype.itemsize == 16 else (keys * min(stretch, 1 << 16)).astype(numpy.int32)
    a['value'] = numpy.arange(len(keys)) % (1 << 24)
    return a


DTYPES = pytest.mark.parametrize("dtype", [workloads.REC8, workloads.REC16I], ids=["8B", "16B"])


@DTYPES
@pytest.mark.parametrize("times", [20, 33, 34, 40, 66, 150, 600])
@pytest.mark.parametrize("form", [0, 2])
def test_every_value_many_times(dtype, times, form):
    """up to 270 bins of one value in a workgroup"""
    sizes = numpy.array(SIZES, numpy.int64)
    a = numpy.concatenate([records(dtype, repeated(n, times, n + times), 1 << (40 if n % 2 else 0)) for n in SIZES])
    g, info = _plan_sort(a, sizes, form)
    assert numpy.array_equal(g, expected(a, sizes))


@DTYPES
@pytest.mark.parametrize("share", [0.1, 0.5, 0.9, 0.99])
@pytest.mark.parametrize("gap", [1, 1 << 12, 1 << 30])
def test_heavy_key_among_others(dtype, share, gap):
    """one key of many records between close and far neighbours"""
    sizes = numpy.array(SIZES * 2, numpy.int64)
    g = numpy.random.default_rng(int(share * 100) + gap % 97)
    parts = []
    for n in sizes:
        k = g.integers(-(1 << 20), 1 << 20, n)
        k[g.random(n) < share] = 77
        near = g.random(n) < 0.02
        k[near] = 77 + g.integers(-2, 3, near.sum())
        parts.append(records(dtype, k, min(gap, 1 << 10) if dtype.itemsize == 8 else gap))
    a = numpy.concatenate(parts)
    out, info = _plan_sort(a, sizes, 0)
    assert numpy.array_equal(out, expected(a, sizes))


@pytest.mark.parametrize("itemsize", [8, 16])
@pytest.mark.parametrize("n", [300007, 2000003, 5000011])
@pytest.mark.parametrize("times", [34, 70, 150, 2000])
def test_sorts_of_repeated_values(itemsize, n, times):
    """the bucket sorts of the one- and two-level forms"""
    P = 5
    k = repeated(n, times, n + times).astype(numpy.uint64) * numpy.uint64((1 << 62) // (n // times + 1))
    a = workloads.records16(k) if itemsize == 16 else k
    check_parity(a, ragged(n, P, 1), ragged(n, P, 2), 'key' if itemsize == 16 else None, device=True)


def plan_ms(a, sizes):
    d, o = lib.mpsort_gpu_dmalloc(a.nbytes), lib.mpsort_gpu_dmalloc(a.nbytes)
    try:
        _lib.check(lib.mpsort_gpu_memcpy_h2d(d, a.ctypes.data, a.nbytes))
        plan = segments.SegmentPlan()
        plan.add(d, o, sizes, a.dtype, 'key')
        ms = min(plan.run() for _ in range(6))
        plan.close()
        g = numpy.empty_like(a)
        _lib.check(lib.mpsort_gpu_memcpy_d2h(g.ctypes.data, o, a.nbytes))
    finally:
        lib.mpsort_gpu_dfree(d)
        lib.mpsort_gpu_dfree(o)
    assert numpy.array_equal(g, expected(a, numpy.array(sizes)))
    return ms


@DTYPES
@pytest.mark.parametrize("size, count", [(500, 100), (1000, 100)])
@pytest.mark.parametrize("share", [0.5, 0.9])
def test_small_segments_with_a_heavy_key_take_little_longer(dtype, size, count, share):
    n = size * count
    g = numpy.random.default_rng(size)
    k = g.integers(0, 1 << 30, n)
    base = plan_ms(records(dtype, k, 1), [size] * count)
    k[g.random(n) < share] = 1 << 29
    ms = plan_ms(records(dtype, k, 1), [size] * count)
    note("distinct %.3f ms, %d%% of one key %.3f ms" % (base, 100 * share, ms))
    assert ms < 2.5 * base


def test_large_segments_of_repeated_values_take_little_longer():
    """100 segments of 100,000 x 8 B, each value 24 times: bins of somewhat
    more than 32 records are no reason to sort a group twice"""
    size, count = 100000, 100
    g = numpy.random.default_rng(1)
    base = plan_ms(records(workloads.REC8, g.integers(0, 1 << 30, size * count), 1), [size] * count)
    ms = plan_ms(records(workloads.REC8, g.integers(0, 4096, size * count), 1), [size] * count)
    note("distinct %.3f ms, 4096 values %.3f ms" % (base, ms))
    assert ms < 2.1 * base
