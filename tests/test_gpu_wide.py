"""The sort of up to 64 ranks in two partition levels (above one partition's
4.3 M records): bytes and counts against the oracle at the edges of its tiles
and buckets, on keys that strain the sampled boundaries, and on every record
type that it takes."""
import sys

import numpy
import pytest

from mpsort import _lib, workloads
from mpsort._lib import lib
from test_gpu_direct import ragged
from test_gpu_histsort import check_parity
from test_gpu_plain_merged import keys

pytestmark = pytest.mark.gpu

N = 4300801  # the smallest size above one partition


@pytest.fixture(autouse=True)
def no_options():
    lib.mpsort_mpi_unset_options(-1)


def note(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("n", [N, 8192 * 526, 8192 * 526 + 1, (1 << 17) * 34 - 1, 9000011])
@pytest.mark.parametrize("P", [1, 5, 64])
def test_sizes(n, P):
    a = workloads.records16(keys("random", n, n % 97))
    note("wide n=%d P=%d" % (n, P))
    out, st = check_parity(a, ragged(n, P, 1), ragged(n, P, 2), 'key', device=True)
    assert st.buckets > 1024 and st.first_passes == 0 and st.second_passes == 0


@pytest.mark.parametrize("shape", ["heavy", "few", "zero_heavy", "sorted", "reversed", "narrow", "two_scales"])
@pytest.mark.parametrize("P", [2, 63])
def test_shapes(shape, P):
    n = N + 12345
    a = workloads.records16(keys(shape, n, 5 + P))
    note("wide shape=%s P=%d" % (shape, P))
    check_parity(a, ragged(n, P, 3), ragged(n, P, 4), 'key', device=True)


@pytest.mark.parametrize("value", [0, 1, 2 ** 64 - 1])
def test_one_key_value(value):
    n, P = N + 7, 3
    k = numpy.full(n, value, numpy.uint64)
    check_parity(workloads.records16(k), ragged(n, P, 5), ragged(n, P, 6), 'key', device=True)
    k[n // 2] = numpy.uint64(value - 1 if value > 1 else value + 1)
    check_parity(workloads.records16(k), ragged(n, P, 5), ragged(n, P, 6), 'key', device=True)


@pytest.mark.parametrize("dt", ["u8", "i8", "i4pair", "keytail", "rows24", "rows40"])
def test_record_types(dt):
    """8- and 16-byte records, signed keys, a key behind its payload, packed
    records of other sizes"""
    n, P = N + 1001, 9
    g = numpy.random.default_rng(8)
    if dt in ("u8", "i8"):
        i = numpy.iinfo(dt)
        a, f = g.integers(i.min, i.max, n, dtype=dt, endpoint=True), None
    else:
        t = {"i4pair": [('key', 'i4'), ('v', 'f4')], "keytail": [('v', 'i8'), ('key', 'i8')],
             "rows24": [('v', 'i8', 2), ('key', 'u8')], "rows40": [('key', 'i4'), ('v', 'i4', 9)]}[dt]
        a, f = numpy.zeros(n, t), 'key'
        i = numpy.iinfo(a['key'].dtype)
        a['key'] = g.integers(i.min, i.max, n, dtype=a['key'].dtype, endpoint=True)
        a['v'] = numpy.arange(n).reshape((n,) + (1,) * (a['v'].ndim - 1))
    check_parity(a, ragged(n, P, 7), ragged(n, P, 8), f, device=True)


def test_buckets_the_sample_misses():
    """every sampled position of one key, so that all other keys share a coarse
    bucket of more tiles than a fine bucket gathers from: the general path
    takes the call, also in place"""
    n, P, S = 256 * 8192 + N, 2, 2048
    u = numpy.arange(S, dtype=numpy.int64)
    k = numpy.random.default_rng(3).integers(1 << 20, 1 << 62, n).astype(numpy.uint64)
    k[(2 * u + 1) * n // (2 * S)] = 5
    a = workloads.records16(k)
    want = a[numpy.argsort(a['key'], kind='stable')]
    out, st = check_parity(a, ragged(n, P, 9), ragged(n, P, 10), 'key', device=True)
    assert numpy.array_equal(out, want)


def test_oversized_fine_buckets():
    """pairs of neighbouring keys, each pair far above the in-LDS capacity,
    spread so that a boundary falls between few of them"""
    n, P = N + 99, 8
    g = numpy.random.default_rng(11)
    k = g.integers(0, 64, n).astype(numpy.uint64) << numpy.uint64(40)
    k += (g.random(n) < 0.01).astype(numpy.uint64)
    check_parity(workloads.records16(k), ragged(n, P, 11), ragged(n, P, 12), 'key', device=True)


def test_in_place_and_overlapping():
    import ctypes
    from gpu_util import even, key_desc
    n, P = N + 5, 4
    a = workloads.records16(keys("heavy", n, 3))
    want = a[numpy.argsort(a['key'], kind='stable')]
    for shift in (0, 1024):
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


@pytest.mark.parametrize("per", [900, 1500, 3500])
def test_groups_of_one_value(per):
    """each key repeated about per times: most fine buckets hold one value and
    stand alone, more of them than the grid of the groups' sorts has
    workgroups, between groups of the values that share a boundary"""
    n, P = N + 999, 7
    g = numpy.random.default_rng(per)
    v = g.integers(0, 2 ** 64, n // per, dtype=numpy.uint64)
    check_parity(workloads.records16(v[g.integers(0, len(v), n)]), ragged(n, P, 8), ragged(n, P, 9), 'key', device=True)
