"""Timed cases of the histogram sort: the calls a program makes through the
public entry points, over the sizes, record types and key distributions of
the repository's benchmark, tests and measured workloads.

A case is a dict of plain values.  ``kind`` names the entry point:

``sort``     mpsort_gpu_newarray on device memory (the plain path), out of place
``learned``  mpsort_gpu_newarray_learned with a model that the program keeps
``batched``  SegmentPlan.run: many independent segments, two record types
``host``     mpsort.sort on numpy arrays (the Python face, host memory)
``train``    learned.train on the output of one plain sort
"""
import ctypes
import math
import os
import sys

import numpy
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mp-sort_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import mpsort  # noqa: E402
from mpsort import _lib, learned, segments  # noqa: E402
from mpsort._lib import KeyDesc, check, lib  # noqa: E402

# record type: bytes per record, key byte offset, key width, signed
RECORDS = {
    "rec16": (16, 0, 8, 0),      # {u64 key, i64 index}: the benchmark's record
    "rec16_tail": (16, 8, 8, 1), # {i64 value, i64 key}: a signed key behind its payload
    "rec8": (8, 0, 4, 1),        # {i32 key, f32 value}
    "key8": (8, 0, 8, 0),        # bare u64 keys
    "particle32": (32, 0, 8, 0), # {u64 id, f32 pos[3], f32 vel[3]}
}
DISTS = ("uniform", "clustered", "lognormal", "zipf", "nearly_sorted", "few")


def listed():
    return [
        # the smallest call in use: the smoke sort, four ranks of 1024 records
        # (a catalogue of a few thousand haloes); launches and waits dominate
        {"name": "sort_4x1024", "kind": "sort", "n": 4096, "ranks": 4, "rec": "rec16", "dist": "uniform",
         "ragged": False},
        # a small array with repeated keys on ragged ranks, signed keys behind
        # their payload: the Python tests' struct arrays
        {"name": "sort_7_ragged_20011", "kind": "sort", "n": 20011, "ranks": 7, "rec": "rec16_tail", "dist": "few",
         "ragged": True},
        # 64 ranks x 65,536 records: the reference benchmark's many-rank run
        # at a size where every rank is small
        {"name": "sort_64x65536", "kind": "sort", "n": 64 * 65536, "ranks": 64, "rec": "rec16", "dist": "uniform",
         "ragged": False},
        # 4 ranks x 1,000,000 uniform keys: the reference's own default run
        {"name": "sort_4x1000000", "kind": "sort", "n": 4000000, "ranks": 4, "rec": "rec16", "dist": "uniform",
         "ragged": False},
        # 8-byte {i32 key, f32 value} records with duplicate-heavy keys, an odd
        # count on ragged ranks
        {"name": "sort_8_rec8_zipf_10000019", "kind": "sort", "n": 10000019, "ranks": 8, "rec": "rec8",
         "dist": "zipf", "ragged": True},
        # particles of 32 bytes put into id order (snapshot matching)
        {"name": "sort_16_particles_12000017", "kind": "sort", "n": 12000017, "ranks": 16, "rec": "particle32",
         "dist": "nearly_sorted", "ragged": False},
        # the benchmark: 2^28 clustered Morton keys on 64 ranks
        {"name": "sort_64x4M_clustered", "kind": "sort", "n": 1 << 28, "ranks": 64, "rec": "rec16",
         "dist": "clustered", "ragged": False},
        # the learned path on another realisation of the field it was trained on
        {"name": "learned_64x1M_clustered", "kind": "learned", "n": 1 << 26, "ranks": 64, "rec": "rec16",
         "dist": "clustered", "ragged": False},
        # the batched workload: segment sizes log-uniform over four decades,
        # half {i32, f32} and half {i64, i64} records, replayed as a graph
        {"name": "batched_2000_mixed", "kind": "batched", "n": 1 << 26, "nseg": 2000, "decades": 4.0},
        # many small segments (groups of one halo each), all sorted in LDS
        {"name": "batched_20000_small", "kind": "batched", "n": 10000000, "nseg": 20000, "decades": 1.0},
        # host arrays through the Python face: 40-byte rows with a two-word
        # radix on 12 ranks (the shape of the reference's issue-7 test)
        {"name": "host_12_rows40_1000003", "kind": "host", "n": 1000003, "ranks": 12},
        # training the key model of the learned path, once per field
        {"name": "train_262144", "kind": "train", "n": 1 << 22, "nsample": 1 << 18, "dist": "clustered"},
    ]


def _log_size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sort"] * 7 + ["learned"] * 2 + ["batched"] * 2 + ["host", "train"])
    if kind == "batched":
        n = _log_size(rng, 200000, 1 << 26)
        nseg = max(2, min(_log_size(rng, 10, 20000), n // 200))
        return {"kind": kind, "n": n, "nseg": nseg, "decades": round(rng.uniform(0.5, 4.0), 2)}
    if kind == "host":
        return {"kind": kind, "n": _log_size(rng, 1000, 2000000), "ranks": rng.randint(1, 64)}
    if kind == "train":
        n = _log_size(rng, 1 << 20, 1 << 24)
        return {"kind": kind, "n": n, "nsample": _log_size(rng, 1 << 14, 1 << 19), "dist": rng.choice(DISTS[:4])}
    rec = rng.choice(["rec16"] * 4 + ["rec16_tail", "rec8", "key8", "particle32"])
    lo, hi = (1 << 20) if kind == "learned" else (1 << 10), (1 << 26) if rec == "particle32" else (1 << 27)
    if kind == "learned":
        rec = rng.choice(["rec16", "rec16", "key8"])
    # ranks as the reference runs them: one, a few, one or two nodes
    ranks = rng.choice([1, 2, 4, 7, 8, 12, 16, 24, 32, 48, 64, 64, 96])
    if kind == "learned":
        ranks = min(ranks, 64)
    return {"kind": kind, "n": _log_size(rng, lo, hi), "ranks": ranks, "rec": rec, "dist": rng.choice(DISTS),
            "ragged": rng.random() < 0.5}


# ---- inputs -----------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed & 0x7FFFFFFFFFFFFFFF)
    return g


def _spread3(v):
    for sh, m in ((32, 0x001F00000000FFFF), (16, 0x001F0000FF0000FF), (8, 0x100F00F00F00F00F),
                  (4, 0x10C30C30C30C30C3), (2, 0x1249249249249249)):
        v = (v | (v << sh)) & m
    return v


def _clustered(n, g, field):
    """Morton keys of Gaussian clumps over a uniform background: 2^16 clumps of
    log-normal radii, 30% background, 21 bits per axis, periodic box."""
    f = _gen(field)
    centre = torch.rand(1 << 16, 3, generator=f, device="cuda", dtype=torch.float64)
    radius = 2.0 ** -8 * torch.exp(torch.randn(1 << 16, generator=f, device="cuda", dtype=torch.float64))
    keys = torch.empty(n, dtype=torch.int64, device="cuda")
    for at in range(0, n, 1 << 25):
        m = min(n - at, 1 << 25)
        c = torch.randint(0, 1 << 16, (m,), generator=g, device="cuda")
        lone = torch.rand(m, generator=g, device="cuda") < 0.3
        k = torch.zeros(m, dtype=torch.int64, device="cuda")
        for axis in range(3):
            x = centre[c, axis] + radius[c] * torch.randn(m, generator=g, device="cuda", dtype=torch.float64)
            u = torch.rand(m, generator=g, device="cuda", dtype=torch.float64)
            x = torch.where(lone, u, x)
            q = torch.clamp(((x - torch.floor(x)) * 2097152.0).to(torch.int64), 0, 2097151)
            k |= _spread3(q) << axis
        keys[at:at + m] = k
    return keys


def _mix64(z):
    def shr(v, s):
        return (v >> s) & ((1 << (64 - s)) - 1)

    z = (z ^ shr(z, 30)) * (0xBF58476D1CE4E5B9 - (1 << 64))
    z = (z ^ shr(z, 27)) * (0x94D049BB133111EB - (1 << 64))
    return z ^ shr(z, 31)


def _keys(dist, n, g, field):
    """n 64-bit keys (an int64 tensor holding the bits)"""
    if dist == "clustered":
        return _clustered(n, g, field)
    if dist == "lognormal":
        mu = torch.tensor([4.0, 9.0, 14.0, 19.0, 24.0, 29.0, 34.0, 39.0], device="cuda", dtype=torch.float64)
        sg = torch.tensor([0.3, 0.5, 0.8, 1.0, 0.6, 0.4, 1.2, 0.7], device="cuda", dtype=torch.float64)
        c = torch.randint(0, 8, (n,), generator=g, device="cuda")
        z = torch.randn(n, generator=g, device="cuda", dtype=torch.float64)
        return torch.exp(mu[c] + sg[c] * z).clamp(max=9.0e18).to(torch.int64)
    if dist == "zipf":
        w = torch.arange(1, (1 << 20) + 1, device="cuda", dtype=torch.float64) ** -1.1
        cdf = torch.cumsum(w, 0)
        u = torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * cdf[-1]
        return _mix64(torch.searchsorted(cdf, u).clamp(max=(1 << 20) - 1) + 1)
    if dist == "nearly_sorted":
        k = torch.arange(n, device="cuda", dtype=torch.int64) * ((1 << 63) // max(n, 1))
        m = n // 200
        if m:
            a = torch.randperm(n, generator=g, device="cuda")[:2 * m]
            k[a] = k[a.roll(m)]
        return k
    if dist == "few":
        return torch.randint(0, 1000, (n,), generator=g, device="cuda") * (3 << 40)
    return torch.randint(-(1 << 63), (1 << 63) - 1, (n,), generator=g, device="cuda")


def _records(rec, keys, g):
    """the records as a tensor whose rows are one record each"""
    n = keys.numel()
    if rec == "key8":
        return keys
    if rec == "rec8":
        out = torch.empty(n, 2, dtype=torch.int32, device="cuda")
        out[:, 0] = (keys >> 20).to(torch.int32)
        out[:, 1] = torch.arange(n, device="cuda", dtype=torch.int32)
        return out
    if rec == "particle32":
        out = torch.randint(0, 1 << 62, (n, 4), generator=g, device="cuda")
        out[:, 0] = keys
        return out
    out = torch.empty(n, 2, dtype=torch.int64, device="cuda")
    k = 1 if rec == "rec16_tail" else 0
    out[:, k] = keys
    out[:, 1 - k] = torch.arange(n, device="cuda", dtype=torch.int64)
    return out


def _cuts(n, P, seed):
    """P counts that add up to n, cut at random places"""
    at = numpy.sort(numpy.random.default_rng(seed).integers(0, n + 1, P - 1))
    return [int(x) for x in numpy.diff(numpy.concatenate([[0], at, [n]]))]


def _even(n, P):
    return [n * (t + 1) // P - n * t // P for t in range(P)]


def _counts(case, seed):
    n, P = case["n"], case["ranks"]
    if not case["ragged"]:
        return _even(n, P), _even(n, P)
    return _cuts(n, P, seed), _cuts(n, P, seed + 1)


def _c_counts(c):
    return (ctypes.c_int64 * len(c))(*c)


def _prepare_device(case, seed):
    g = _gen(seed)
    size, off, width, signed = RECORDS[case["rec"]]
    a = _records(case["rec"], _keys(case["dist"], case["n"], g, seed + 7), g)
    nin, nout = _counts(case, seed)
    return {"case": case, "in": a, "out": torch.empty_like(a), "nin": _c_counts(nin), "nout": _c_counts(nout),
            "P": len(nin), "size": size,
            "key": KeyDesc(offset=off, width=width, is_signed=signed, nwords=1, reserved=0)}


def _plain(st):
    check(lib.mpsort_gpu_newarray(st["in"].data_ptr(), st["nin"], st["P"], st["out"].data_ptr(), st["nout"],
                                  st["size"], ctypes.byref(st["key"]), _lib.DEVICE_PTRS))
    return st["out"]


def _prepare_train(case, seed):
    g = _gen(seed)
    keys = _keys(case["dist"], case["n"], g, seed + 7)
    a = _records("rec16", keys, g)
    a[:, 0] &= (1 << 63) - 1  # torch sorts signed integers
    order = torch.sort(a[:, 0], stable=True).indices
    return {"case": case, "in": a[order].contiguous(), "seed": 1 + seed % 1000,
            "key": KeyDesc(offset=0, width=8, is_signed=0, nwords=1, reserved=0)}


def _prepare_batched(case, seed):
    g = _gen(seed)
    r = numpy.random.default_rng(seed)
    nseg, n = case["nseg"], case["n"]
    st = {"case": case, "in": [], "out": [], "plan": segments.SegmentPlan(graph=True)}
    for count, m, dtype in ((nseg // 2, n // 2, numpy.dtype([("key", "<i4"), ("value", "<f4")])),
                            (nseg - nseg // 2, n - n // 2, numpy.dtype([("key", "<i8"), ("value", "<i8")]))):
        # log-uniform sizes, rescaled; the largest takes what rounding left
        raw = 10.0 ** (r.random(count) * case["decades"])
        half = numpy.maximum(1, numpy.floor(raw * (m - count) / raw.sum())).astype(numpy.int64)
        half[numpy.argmax(half)] += m - half.sum()
        k = _keys("uniform", m, g, seed)
        a = _records("rec8" if dtype.itemsize == 8 else "rec16", k, g)
        st["in"].append(a)
        st["out"].append(torch.empty_like(a))
        st["plan"].add(a.data_ptr(), st["out"][-1].data_ptr(), half, dtype, "key")
    return st


ROWS40 = numpy.dtype([("radix", "<u8", (2,)), ("ext", "<u8", (3,))])


def _prepare_host(case, seed):
    r = numpy.random.default_rng(seed)
    n = case["n"]
    a = numpy.empty(n, ROWS40)
    a["radix"][:, 0] = r.integers(0, 2 ** 64, n, dtype=numpy.uint64)
    a["radix"][:, 1] = r.integers(0, 1000, n)  # the most significant word: many ties
    a["ext"] = r.integers(0, 2 ** 63, (n, 3))
    return {"case": case, "in": a, "out": numpy.empty_like(a), "comm": mpsort.VirtualComm(vranks=case["ranks"])}


def prepare(case, seed):
    """What the calling program has in hand: inputs on the GPU (host arrays for
    the Python face), its rank counts, the plan or the model it keeps."""
    kind = case["kind"]
    if kind == "host":
        return _prepare_host(case, seed)
    if kind == "train":
        st = _prepare_train(case, seed)
    elif kind == "batched":
        st = _prepare_batched(case, seed)
    else:
        st = _prepare_device(case, seed)
        if kind == "learned":
            # the model of another realisation of the same distribution
            g = _gen(seed + 1)
            other = _keys(case["dist"], case["n"], g, seed + 7)
            t = dict(st)
            t["in"] = _records(case["rec"], other, g)
            torch.cuda.synchronize()
            srt = _plain(t)
            k = st["key"]
            st["model"] = learned.train(None, nsample=1 << 18, seed=3,
                                        device_ptr=(srt.data_ptr(), case["n"], st["size"], k))
    torch.cuda.synchronize()  # the library works on a stream of its own
    return st


# ---- one pass ---------------------------------------------------------------
def run(st):
    kind = st["case"]["kind"]
    if kind == "sort":
        return _plain(st)
    if kind == "learned":
        check(lib.mpsort_gpu_newarray_learned(st["in"].data_ptr(), st["nin"], st["P"], st["out"].data_ptr(),
                                              st["nout"], st["size"], ctypes.byref(st["key"]), st["model"]._h,
                                              _lib.DEVICE_PTRS))
        return st["out"]
    if kind == "batched":
        st["plan"].run()
        return st["out"]
    if kind == "host":
        mpsort.sort(st["in"], "radix", st["out"], comm=st["comm"])
        return st["out"].view("<i8").reshape(len(st["out"]), 5)
    model = learned.train(None, nsample=st["case"]["nsample"], seed=st["seed"],
                          device_ptr=(st["in"].data_ptr(), st["case"]["n"], 16, st["key"]))
    raw, leaves = model.params()
    model.close()
    return raw, leaves


def exact(case, seed):
    # sorted records are whole numbers, and weights after Adam steps have no
    # value that 64-bit arithmetic would settle
    return None


def work(case):
    """every record read once and written once; training reads its sample and
    passes 1/16 of it through the 1-32-32-1 network forward and backward in
    each of 2000 steps"""
    n = case["n"]
    if case["kind"] == "train":
        s = case["nsample"]
        return {"bytes": 16 * s, "flops": 2000 * (s // 16) * 6 * (32 + 32 * 32 + 32)}
    if case["kind"] == "batched":
        return {"bytes": 2 * (n // 2) * (8 + 16), "flops": 0}
    if case["kind"] == "host":
        return {"bytes": 2 * n * ROWS40.itemsize, "flops": 0}
    return {"bytes": 2 * n * RECORDS[case["rec"]][0], "flops": 0}
