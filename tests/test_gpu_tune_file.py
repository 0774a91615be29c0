"""The tuning file: a choice is read when it was made for this set of plans, and
one of another version of the library (no number, or another) is not."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = """
import sys
sys.path[:0] = [%r, %r]
import numpy
from mpsort import segments, workloads
from mpsort._lib import lib
from test_gpu_segments import expected, make
sizes = [500] * 300
a = make(workloads.REC16I, sizes, 5)
d = lib.mpsort_gpu_dmalloc(a.nbytes)
assert lib.mpsort_gpu_memcpy_h2d(d, a.ctypes.data, a.nbytes) == 0
p = segments.SegmentPlan(tune=True)
p.add(d, d, sizes, a.dtype, 'key')
p.run()
print("THRESHOLD", p.info()["threshold"], flush=True)
p.close()
lib.mpsort_gpu_dfree(d)
""" % (os.path.join(ROOT, "mp-sort_amd"), os.path.join(ROOT, "tests"))


@pytest.mark.parametrize("prefix, read", [("", False), ("plans=1 ", False), ("plans=2 ", True)])
def test_choices_of_other_plans_are_not_read(prefix, read, tmp_path):
    """a choice that no tuning makes: all segments of 500 records above the
    in-LDS threshold"""
    f = tmp_path / "tune.txt"
    f.write_text(prefix + "rw=4 keybytes=8 class=8 block=256 items=16 threshold=0 form=0\n")
    r = subprocess.run([sys.executable, "-c", CHILD], env=dict(os.environ, MPSORT_GPU_TUNE_CACHE=str(f)),
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    threshold = int(r.stdout.split("THRESHOLD")[1])
    assert (threshold == 0) == read
    assert f.read_text().startswith("plans=2 rw=4 keybytes=8 class=8 ")
    assert len(f.read_text().splitlines()) == 1
