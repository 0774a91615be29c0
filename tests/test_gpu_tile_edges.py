"""The two-level sort at the edges of its tiles of 6144 records and of its
offset rows, which are padded to 64 tiles and hold one entry past the last:
full and nearly full last tiles, one record more, ranks of whole tiles, and
ranks without records."""
import numpy
import pytest

from mpsort import _lib, workloads
from mpsort._lib import lib
from test_gpu_direct import note
from test_gpu_histsort import check_parity
from test_gpu_plain_merged import keys

pytestmark = pytest.mark.gpu

TILE = 6144
LEAST = 4300800 // TILE + 1  # tiles of the smallest call, 701


@pytest.fixture(autouse=True)
def no_options():
    lib.mpsort_mpi_unset_options(-1)


def check(a, nin, nout, field='key'):
    out, st = check_parity(a, nin, nout, field, device=True)
    assert st.form == _lib.FORM_TWO_LEVELS


@pytest.mark.parametrize("itemsize, n", [(16, t * TILE + d) for t in (LEAST, 703, 704) for d in (-1, 0, 1)] +
                         [(8, t * TILE + d) for t in (704, 768) for d in (0, 1)])
def test_one_rank(itemsize, n):
    """703, 704 and 705 tiles: the entry past the last is the last of its row
    of 64, the first of another, and the second"""
    note("tile edges n=%d itemsize=%d" % (n, itemsize))
    k = keys("heavy", n, n % 89)
    a = workloads.records16(k) if itemsize == 16 else k
    check(a, [n], [n], 'key' if itemsize == 16 else None)


@pytest.mark.parametrize("tiles", [[700, 4], [64, 64, 640, 0, 0], [0, 703, 1], [0, 0, 705], [1] * 63 + [641], [704, 0]])
def test_ranks_of_whole_tiles(tiles):
    """and empty ranks, the first and the last among them"""
    nin = numpy.array(tiles, numpy.int64) * TILE
    n, P = int(nin.sum()), len(tiles)
    g = numpy.random.default_rng(P)
    nout = numpy.diff(numpy.concatenate([[0], numpy.sort(g.integers(0, n + 1, P - 1)), [n]]))
    a = workloads.records16(keys("random", n, P))
    check(a, nin, nout)
    check(a, nin, nin[::-1].copy())


@pytest.mark.parametrize("d", [-1, 1])
def test_ranks_of_a_record_more_or_less(d):
    nin = numpy.array([100 * TILE + d, 64 * TILE, d + 1, 540 * TILE - d, 2 + d], numpy.int64)
    n = int(nin.sum())
    check(workloads.records16(keys("two_scales", n, 3)), nin, nin[::-1].copy())
