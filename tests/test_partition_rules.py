"""The sizes up to which a call takes the two-level partition, against the
distribution of its sampled buckets (CPU only; the constants are read from the
sources)."""
import os
import re

import pytest
from scipy.stats import beta

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mp-sort_amd", "csrc")


def constants():
    c = {}
    for name in ("lsort.h", "direct.h", "wide.h", "api.cpp"):
        text = open(os.path.join(CSRC, name)).read()
        for k, v in re.findall(r"^constexpr \w+ (k\w+) = ([^;]+);", text, re.M):
            v = re.sub(r"\(\w+_t\)", "", v).replace("/", "//")
            try:
                c[k] = eval(v, {"__builtins__": {}}, dict(c))
            except (NameError, SyntaxError):
                pass
    return c


C = constants()


def chance_of_a_missed_bucket(n):
    """of a call with randomly ordered distinct keys: an upper bound of the
    chance that some coarse bucket has more tiles than a fine bucket gathers
    from.  The records between two boundaries that are s of S sample keys
    apart are a share of all that follows Beta(s, S - s + 1)."""
    W = min(C["kWideBuckets"], max(2, -(-n // C["kWideCoarse"])))
    S = min(C["kDirectMaxChunks"], -(-32 * W // C["kDirectChunk"])) * C["kDirectChunk"]
    s = S // W
    return W * beta.sf(C["kWideRuns"] * C["kWideTile"] / n, s, S - s + 1)


@pytest.mark.parametrize("share", [1.0, 0.9, 0.76, 0.5, 0.1, 0.013])
def test_the_two_level_sort_reaches_its_largest_size(share):
    n = int(C["kWideMaxRecords"] * share)
    assert n > C["kDirectMaxRecords"]
    assert chance_of_a_missed_bucket(n) < 2e-5


def test_the_chance_is_not_small_beyond():
    assert chance_of_a_missed_bucket(400000000) > 1e-3
    assert chance_of_a_missed_bucket(1 << 29) > 0.9
