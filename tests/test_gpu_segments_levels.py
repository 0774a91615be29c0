"""The batched sort's workgroup sizes for small segments and its partition
level for segments above the in-LDS sizes: both record types at the edges of
the sizes, duplicate-heavy keys, keys whose sample misses a bucket's weight,
and graph replays against per-segment stable sorts."""
import numpy
import pytest

from mpsort import _lib, segments, workloads
from mpsort._lib import lib
from test_gpu_segments import expected, make, note, _plan_sort

pytestmark = pytest.mark.gpu

LEVEL = 512 * 1843  # the largest segment of one partition level
SIZES = [1, 2, 63, 64, 65, 127, 128, 767, 768, 769, 1535, 1536, 1537, 3072, 3073, 4607, 4608, 4609, 9215, 9216, 9217,
         0, 6144 * 2 - 1, 6144 * 2, 6144 * 2 + 1, 100003, LEVEL - 1, LEVEL, LEVEL + 1]


@pytest.mark.parametrize("dtype", [workloads.REC8, workloads.REC16I], ids=["8B", "16B"])
@pytest.mark.parametrize("key_bits", [None, 40, 34, 3], ids=["spread", "dup40", "dup34", "dup3"])
@pytest.mark.parametrize("form", [0, 2])
def test_size_edges(dtype, key_bits, form):
    sizes = numpy.array(SIZES, numpy.int64)
    a = make(dtype, sizes, 5 + form, key_bits=key_bits)
    note("segment levels %s keybits %s form %d" % (dtype, key_bits, form))
    g, info = _plan_sort(a, sizes, form)
    assert info["large_segments"] == sum(1 for s in SIZES if s > 9216)
    assert numpy.array_equal(g, expected(a, sizes))


@pytest.mark.parametrize("dtype", [workloads.REC8, workloads.REC16I], ids=["8B", "16B"])
def test_the_sample_misses_the_weight(dtype):
    """every sampled position of one key: the other keys share a bucket above
    the in-LDS capacity, sorted without a count taken to the host; replayed
    on new contents, with eager work between the replays"""
    sizes = numpy.array([100003, 700, 60001], numpy.int64)
    d = lib.mpsort_gpu_dmalloc(int(sizes.sum()) * dtype.itemsize)
    o = lib.mpsort_gpu_dmalloc(int(sizes.sum()) * dtype.itemsize)
    plan = segments.SegmentPlan(graph=True)
    try:
        for rep in range(4):
            a = make(dtype, sizes, 31 + rep)
            if rep != 2:
                b = 0
                for n in sizes:
                    m = min(4096, int(n))
                    u = numpy.arange(m, dtype=numpy.int64)
                    a['key'][b + (2 * u + 1) * n // (2 * m)] = -7
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


@pytest.mark.parametrize("graph", [False, True])
def test_groups_that_depend_on_each_other(graph):
    """the second group reads what the first wrote: the parts of a plan run
    side by side only where their buffers are apart"""
    dtype = workloads.REC16I
    sizes = numpy.array([300, 20000, 5, 1000, 60001], numpy.int64)
    n = int(sizes.sum())
    a = make(dtype, sizes, 77, key_bits=16)
    d = [lib.mpsort_gpu_dmalloc(a.nbytes) for _ in range(3)]
    plan = segments.SegmentPlan(graph=graph)
    try:
        _lib.check(lib.mpsort_gpu_memcpy_h2d(d[0], a.ctypes.data, a.nbytes))
        plan.add(d[0], d[1], sizes, dtype, 'key')
        plan.add(d[1], d[2], numpy.array([n], numpy.int64), dtype, 'key')
        for _ in range(3):
            plan.run()
            g = numpy.empty_like(a)
            _lib.check(lib.mpsort_gpu_memcpy_d2h(g.ctypes.data, d[2], a.nbytes))
            assert numpy.array_equal(g, expected(a, [n]))
    finally:
        plan.close()
        for p in d:
            lib.mpsort_gpu_dfree(p)
