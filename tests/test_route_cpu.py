"""The rules by which a 16-bit launch is given to the persistent kernel or to the one with resident tables, and to units of 16 or 32 query
rows there (turbodeberta_amd/csrc/attn_resident.hip), at launches that were measured.  Without a device they count with 256 compute units."""
import ctypes as C
import os
import re

import pytest

from turbodeberta_amd import _lib

CSRC = os.path.join(os.path.dirname(_lib.PKG), "turbodeberta_amd", "csrc")
TYPES = {"const void": C.c_void_p, "void": C.c_void_p, "const int32_t": C.c_void_p, "int64_t": C.c_int64, "int32_t": C.c_int32, "float": C.c_float}


def _params():
    """TdbKernelParams, as tdb_internal.h declares it."""
    body = re.search(r"struct TdbKernelParams \{(.*?)\n\};", open(os.path.join(CSRC, "tdb_internal.h")).read(), re.S).group(1)
    fields = []
    for decl in re.sub(r"//.*", "", body).split(";"):
        m = re.match(r"\s*((?:const )?\w+)\s*(.*)", decl, re.S)
        if m:
            fields += [(n.strip(" *\n"), TYPES[m[1]]) for n in m[2].split(",")]
    return type("TdbKernelParams", (C.Structure,), {"_fields_": fields})


def _rule(name):
    fn = getattr(_lib.load(), f"_Z17tdb_resident_{name}RK15TdbKernelParams")
    fn.argtypes, fn.restype = [C.c_void_p], C.c_bool
    return fn


def _launch(kind, lens, heads=12, terms=2):
    p = _params()()
    p.B, p.H, p.D, p.L, p.span, p.lut_half = len(lens), heads, 64, max(lens), 256, 511
    p.pk, p.pq = (1 if terms > 0 else None), (1 if terms > 1 else None)
    if kind == "packed":
        p.varlen, p.total, p.cu_seqlens = 1, sum(lens), 1
    elif kind == "padded":
        p.seqlens = 1
    return C.byref(p)


def _even(n, lo, hi):
    return [lo + (hi - lo) * i // max(n - 1, 1) for i in range(n)]


SHORT_ONES = [10] * 20 + [100] * 10 + [190] * 13 + [233]               # 83 tokens in the mean


@pytest.mark.parametrize("kind,lens,heads,terms,resident", [
    ("packed", _even(64, 16, 512), 12, 2, True), ("padded", _even(32, 384, 512), 12, 2, True), ("equal", [4096] * 4, 12, 2, True),
    ("packed", _even(8, 1024, 4096), 12, 2, True), ("equal", [250] * 8, 16, 2, False), ("padded", [840, 2100], 12, 2, False),
    ("packed", _even(35, 384, 384), 8, 0, True), ("packed", [298, 1494], 24, 0, True), ("equal", [2048], 8, 0, True),       # no terms: always
])
def test_which_kernel(kind, lens, heads, terms, resident):
    assert _rule("pays")(_launch(kind, lens, heads, terms)) == resident


@pytest.mark.parametrize("kind,lens,heads,resident", [
    ("equal", [1535] * 6, 12, False), ("equal", [1536] * 6, 12, True), ("equal", [1990], 16, False),        # 5.25 and 6 units a round
    ("packed", [2269], 16, True), ("packed", [1717, 1717], 6, False), ("packed", [500, 1700, 1100, 2290], 6, False), ("packed", [1024, 1000, 4000], 8, True),
    ("padded", [900, 1935], 12, False), ("padded", [1935], 12, True), ("padded", [1000, 1700, 400], 12, True),
    # the longest decides alone (52 us there, 69 here), or has far steps enough (118 here, 160 there)
    ("packed", [343, 234, 843, 265, 204, 1064, 259, 74, 2322, 910, 279], 6, False), ("packed", [4603, 509], 8, True), ("packed", [1835, 3059], 12, True),
])
def test_which_kernel_of_long_launches(kind, lens, heads, resident):
    assert _rule("pays")(_launch(kind, lens, heads)) == resident


@pytest.mark.parametrize("kind,lens,heads,resident", [
    ("padded", _even(16, 64, 512), 16, True), ("padded", _even(13, 64, 512), 16, False), ("padded", _even(16, 64, 512), 12, False),
    ("packed", _even(15, 200, 512), 16, True), ("packed", _even(10, 200, 512), 16, False),
    ("packed", [562] + [48] * 39, 16, False), ("packed", [562] + [200] * 39, 16, True),         # a tenth and a third of the longest in the mean
])
def test_which_kernel_of_workgroups_that_keep_one_head(kind, lens, heads, resident):
    assert _rule("pays")(_launch(kind, lens, heads)) == resident


@pytest.mark.parametrize("kind,lens,heads,wide", [
    ("packed", _even(64, 16, 512), 12, True), ("padded", _even(32, 384, 512), 12, True), ("packed", _even(8, 1024, 4096), 12, True),
    ("equal", [512] * 64, 12, True), ("equal", [180], 12, False), ("packed", [300, 200], 12, False),
    ("packed", SHORT_ONES, 12, False), ("packed", _even(32, 19, 195), 8, False), ("packed", [233] * 44, 12, True),          # short texts among longer ones
    ("packed", [1835, 3059], 8, True), ("packed", [100] * 5 + [3059], 8, False),                                            # long ones of similar lengths
    ("packed", _even(66, 22, 222), 8, False),           # a part has half of the tokens
])
def test_which_units(kind, lens, heads, wide):
    assert _rule("wide")(_launch(kind, lens, heads)) == wide


@pytest.mark.parametrize("kind,lens,heads,terms,sets", [
    ("padded", _even(8, 96, 384), 12, 2, 1), ("equal", [128] * 32, 12, 2, 1), ("packed", _even(12, 209, 209), 12, 2, 1),
    ("equal", [512] * 2, 12, 2, 2), ("equal", [256] * 4, 12, 2, 2), ("equal", [190] * 3, 16, 2, 2), ("padded", _even(3, 151, 460), 12, 2, 2),
    ("equal", [128] * 2, 12, 2, 0), ("equal", [512], 12, 2, 0), ("equal", [21] * 44, 12, 2, 0), ("packed", _even(58, 17, 30), 16, 2, 0),
    ("packed", [134] * 7, 12, 1, 0), ("equal", [59] * 8, 16, 1, 0),
    ("packed", [126] + [23] * 12, 12, 2, 0), ("packed", [247] + [32] * 19, 8, 2, 0), ("packed", [247] + [150] * 9, 8, 2, 1),    # a long one among short ones
    ("equal", [68] * 9, 16, 2, 0), ("equal", [120] * 9, 16, 2, 1), ("padded", [139] * 6, 16, 2, 0),
])
def test_which_float32_kernel(kind, lens, heads, terms, sets):
    fn = _lib.load()._Z18tdb_f32_split_setsRK15TdbKernelParams
    fn.argtypes, fn.restype = [C.c_void_p], C.c_int
    assert fn(_launch(kind, lens, heads, terms)) == sets
