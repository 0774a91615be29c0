"""The fault hooks on the calls that are sorted without per-rank steps: data
changed between two steps of a partition is found by the checksum, and buckets
above a forced capacity take the radix path with the same result."""
import numpy
import pytest

from gpu_util import even, gpu_sort, gpu_sort_device, last_counts
from mpsort import _lib, learned, workloads
from mpsort._lib import lib
from test_gpu_direct import note, ragged
from test_gpu_histsort import check_parity
from test_gpu_learned import keys_of, trained
from test_gpu_plain_merged import keys

pytestmark = pytest.mark.gpu

# a size of every form: ranks counted, one workgroup, one level, two levels
FORMS = pytest.mark.parametrize("n, form", [(3000, _lib.FORM_ONE_LAUNCH), (7000, _lib.FORM_ONE_LAUNCH),
                                            (100000, _lib.FORM_ONE_LEVEL), (4400000, _lib.FORM_TWO_LEVELS)])


@pytest.fixture(autouse=True)
def no_options_and_no_faults_after():
    lib.mpsort_mpi_unset_options(-1)
    yield
    _lib.check(lib.mpsort_gpu_set_faults(0, 0))


def faults(bits, cap=0):
    _lib.check(lib.mpsort_gpu_set_faults(bits | _lib.FAULT_KEEP_FORM, cap))


@FORMS
@pytest.mark.parametrize("P", [1, 8])
@pytest.mark.parametrize("rec", ["rec16", "heavy16", "u8", "rows24"])
def test_corruption_is_detected(n, form, P, rec):
    k = keys("heavy" if rec == "heavy16" else "random", n, 3)
    if rec == "u8":
        a, field = k, None  # (the key fills the record: the recorded sum is changed)
    elif rec == "rows24":
        a, field = numpy.zeros(n, [('v', 'i8', 2), ('key', 'u8')]), 'key'
        a['key'] = k
    else:
        a, field = workloads.records16(k), 'key'
    note("corrupt %s n=%d P=%d" % (rec, n, P))
    faults(_lib.FAULT_CORRUPT)
    with pytest.raises(_lib.MPSortError) as e:
        gpu_sort_device(a, ragged(n, P, 1), ragged(n, P, 2), field)
    assert e.value.code == _lib.MPSORT_ERR_CHECKSUM
    # without the checksum nothing is checked
    out, st = gpu_sort_device(a, even(n, P), even(n, P), field, flags=_lib.NO_CHECKSUM)
    assert st.form == form
    _lib.check(lib.mpsort_gpu_set_faults(0, 0))
    out, st = check_parity(a, even(n, P), even(n, P), field, device=True)
    assert st.form == form


@pytest.mark.parametrize("n, form", [(100000, _lib.FORM_ONE_LEVEL), (4400000, _lib.FORM_TWO_LEVELS)])
@pytest.mark.parametrize("cap", [1, 700, 1300])
@pytest.mark.parametrize("rec", ["rec16", "heavy16", "u8", "rows24"])
def test_buckets_above_a_forced_capacity(n, form, cap, rec):
    """the radix path of oversized buckets, up to thousands of them, in and
    out apart and in place"""
    P = 5
    k = keys("heavy" if rec == "heavy16" else "random", n, 4)
    if rec == "u8":
        a, field = k, None
    elif rec == "rows24":
        a, field = numpy.zeros(n, [('v', 'i8', 2), ('key', 'u8')]), 'key'
        a['key'], a['v'] = k, numpy.arange(2 * n).reshape(n, 2)
    else:
        a, field = workloads.records16(k), 'key'
    note("capacity %d %s n=%d" % (cap, rec, n))
    faults(_lib.FAULT_BUCKET_CAP, cap)
    out, st = check_parity(a, ragged(n, P, 1), ragged(n, P, 2), field, device=True)
    assert st.form == form and st.buckets_overflow > 0
    assert cap > 1 or st.buckets_overflow > (20 if form == _lib.FORM_ONE_LEVEL else 2000)
    if cap != 1:
        from test_gpu_histsort import _device_inplace
        got, st = _device_inplace(a, ragged(n, P, 1), field)
        assert st.form == form and st.buckets_overflow > 0
        assert numpy.array_equal(got.view(numpy.uint8), out.view(numpy.uint8))


@pytest.mark.parametrize("bits, cap", [(_lib.FAULT_BUCKET_CAP, 900), (_lib.FAULT_CORRUPT, 0)])
def test_learned_two_levels(bits, cap):
    n, P = 4400000, 16
    model = trained("uniform", n)
    a = workloads.records16(keys_of("uniform", n, 5))
    ref, _ = gpu_sort(a, even(n, P), even(n, P), 'key')
    ref_counts = last_counts(P, 8)
    faults(bits, cap)
    try:
        if bits == _lib.FAULT_CORRUPT:
            with pytest.raises(_lib.MPSortError) as e:
                learned.sort_learned(a, model, 'key', nin=even(n, P))
            assert e.value.code == _lib.MPSORT_ERR_CHECKSUM
            return
        out = learned.sort_learned(a, model, 'key', nin=even(n, P))
        st = _lib.last_stats()
    finally:
        model.close()
    assert st.form == _lib.FORM_TWO_LEVELS and st.buckets_overflow > 0
    assert numpy.array_equal(out, ref)
    counts = last_counts(P, 8)
    for k in ("C", "P", "myCLT", "myCLE", "myC", "send"):
        assert numpy.array_equal(counts[k], ref_counts[k]), k


def test_hooks_without_the_flag_take_the_ranks():
    n = 100000
    a = workloads.records16(keys("random", n, 4))
    _lib.check(lib.mpsort_gpu_set_faults(_lib.FAULT_BUCKET_CAP, 700))
    out, st = check_parity(a, even(n, 4), even(n, 4), 'key', device=True)
    assert st.form == _lib.FORM_RANKS
