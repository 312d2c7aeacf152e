"""cutTable (slang_amd/csrc/cv_permuto_parts.h), the host code that cuts the permutohedral encoder's table gradient into
parts for LDS, compiled by itself and checked for tables of every entry size: no part may exceed a compute unit's LDS,
and the parts cover what every level adds to once."""
import ctypes
import os
import random
import subprocess

import pytest

from slang_amd import _lib

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LDS_DOUBLES = 160 * 1024 // 8

SOURCE = """
#include "cv_permuto_parts.h"
extern "C" int cut(const CvPermutoDesc* d, uint32_t* out, uint32_t* sliced)
{
    cv::TableParts t;
    const bool ok = cv::cutTable(*d, t);
    for (uint32_t p = 0; ok && p < t.count; ++p) {
        const cv::TablePart& q = t.part[p];
        out[4 * p] = q.base; out[4 * p + 1] = q.elems; out[4 * p + 2] = q.first; out[4 * p + 3] = q.end;
    }
    *sliced = ok ? t.sliced : 0;
    return ok ? (int)t.count : -1;
}
extern "C" int beside(uint32_t count, uint32_t elems, uint32_t batch, uint32_t cus, int sliced, uint32_t* groups)
{
    cv::TableParts t{};
    t.count = count;
    t.sliced = sliced;
    for (uint32_t p = 0; p < count; ++p) t.part[p].elems = p + 1 < count ? 1u : elems;
    cv::dealGroups(t, batch, cus);
    *groups = t.groups;
    return cv::positionsBeside(t, batch, cus);
}
// parts and workgroups of a launch (out[4 n ..]: as cut's; returned: n * 65536 + workgroups), spread: cutByLevel may be asked
extern "C" int plan(const CvPermutoDesc* d, uint32_t batch, uint32_t cus, int spread, uint32_t* out)
{
    cv::TableParts t{};
    if (!cv::planTable(*d, batch, cus, spread != 0, t)) return -1;
    for (uint32_t p = 0; p < t.count; ++p) { out[4 * p] = t.part[p].base; out[4 * p + 1] = t.part[p].elems; out[4 * p + 2] = t.part[p].first; out[4 * p + 3] = t.part[p].end; }
    return (int)(t.count * 65536u + t.groups);
}
extern "C" int meet(const uint64_t* a, const uint64_t* b, uint32_t rows) { return cv::rowsMeet({a[0], a[1], a[2]}, {b[0], b[1], b[2]}, rows); }
"""


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    d = tmp_path_factory.mktemp("parts")
    (d / "parts.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(REPO, "include"),
                    "-I", os.path.join(REPO, "slang_amd", "csrc"), "-o", str(d / "parts.so"), str(d / "parts.cpp")], check=True)
    return ctypes.CDLL(str(d / "parts.so"))


@pytest.fixture(scope="module")
def cut(built):
    lib = built

    def call(F, tables):
        """tables: (offset, size) in entries per level; the parts (base, elems, first, end) and `sliced`, or None"""
        desc = _lib.CvPermutoDesc(dimensions=3, featureDimensionPerEntry=F, maxLevels=len(tables), maxLevel=99.0)
        for l, (offset, size) in enumerate(tables):
            lv = desc.levelInfo[l]
            lv.currentLevelIndex, lv.offsetOfFeatureTable, lv.featureTableSize = l, offset, size
        out, sliced = (ctypes.c_uint32 * (4 * 144))(), ctypes.c_uint32()
        n = lib.cut(ctypes.byref(desc), out, ctypes.byref(sliced))
        return None if n < 0 else ([tuple(out[4 * p:4 * p + 4]) for p in range(n)], sliced.value)
    return call


def behind_one_another(sizes):
    return [(sum(sizes[:l]), s) for l, s in enumerate(sizes)]


def check(parts, sliced, F, tables):
    """Every level's elements are covered by its parts once; slices only where `sliced` says so."""
    for base, elems, first, end in parts:
        assert 0 < elems <= LDS_DOUBLES and base % F == 0 and elems % F == 0 and first < end, (F, tables, base, elems)
    for l, (offset, size) in enumerate(tables):
        lo, hi = offset * F, (offset + size) * F
        mine = sorted((base, base + elems) for base, elems, first, end in parts if first <= l < end)
        if len(mine) == 1:
            assert mine[0][0] <= lo and hi <= mine[0][1], (F, tables, l, mine)
        else:
            assert sliced and mine and mine[0][0] == lo and mine[-1][1] == hi, (F, tables, l, mine)
            assert all(a[1] == b[0] for a, b in zip(mine, mine[1:])), (F, tables, l, mine)


@pytest.mark.parametrize("F", range(1, 65))
def test_parts_of_every_entry_size_fit_the_lds(cut, F):
    rng = random.Random(F)
    sizes = [[1 << n] * levels for n in range(0, 21) for levels in (1, 3, 8)]
    sizes += [[s] * 2 for s in (13653, 20480, 20481, 40960, 3 * 4096 + 1)]
    sizes += [[int(2 ** rng.uniform(0, 19)) for _ in range(rng.randint(1, 16))] for _ in range(200)]
    for s in sizes:
        got = cut(F, behind_one_another(s))
        slices = [-(-n // (LDS_DOUBLES // F)) for n in s]
        if max(slices) > 16:
            assert got is None, (F, s)
        elif sum(slices) <= 144:
            assert got is not None, (F, s)
        if got is not None:
            check(*got, F, behind_one_another(s))
            assert sum(e for _, e, _, _ in got[0]) == sum(s) * F


@pytest.mark.parametrize("F", [1, 2, 3, 4, 7, 15, 64])
def test_parts_of_tables_in_any_layout(cut, F):
    # levels with gaps between them, in any order, on the same entries, far apart
    rng = random.Random(100 + F)
    for case in range(400):
        levels, top = rng.randint(1, 16), rng.choice([4, 8, 12, 16])
        sizes = [max(1, int(2 ** rng.uniform(0, top))) for _ in range(levels)]
        tables = behind_one_another(sizes)
        kind = case % 4
        if kind == 0: tables = [(o + 5 * l, s) for l, (o, s) in enumerate(tables)]
        if kind == 1: tables = [(sum(sizes) - o - s, s) for o, s in tables]
        if kind == 2: tables = [(rng.choice(tables)[0], s) for _, s in tables]
        if kind == 3: tables = [(rng.randrange(0, (1 << 32) // F - (1 << 17)), s) for _, s in tables]
        slices = [-(-s // (LDS_DOUBLES // F)) for s in sizes]
        got = cut(F, tables)
        if max(slices) <= 16 and sum(slices) <= 144:
            assert got is not None, (F, tables)
        if got is not None:
            check(*got, F, tables)
    # what fits half of the LDS is one part, which also gives the position gradients
    small = LDS_DOUBLES // 2 // F
    if small >= 8:
        n = small // 4
        for tables in ([(l * n, n - 1) for l in range(4)], [((3 - l) * n, n) for l in range(4)], [(0, n)] * 4, [(7, n), (7 + n, n), (8, 3)]):
            assert cut(F, tables)[0] == [(min(o for o, _ in tables) * F, (max(o + s for o, s in tables) - min(o for o, _ in tables)) * F, 0, len(tables))]
    # elements beyond 32 bits: not cut
    assert cut(F, [(0, 4), ((1 << 32) // F - 2, 4)]) is None


def test_rows_that_meet(built):
    def meet(a, b, rows):
        got = {bool(built.meet((ctypes.c_uint64 * 3)(*x), (ctypes.c_uint64 * 3)(*y), rows)) for x, y in ((a, b), (b, a))}
        assert len(got) == 1
        return got.pop()
    for at in (0x1000, (1 << 48) - 4):
        assert meet((at, 12, 12), (at, 64, 64), 5) and meet((at, 12, 12), (at, 12, 12), 1)
        assert not meet((at, 12, 12), (at + 60, 12, 12), 5) and meet((at, 12, 12), (at + 59, 12, 12), 5)
        assert meet((at, 64, 12), (at + 12, 64, 52), 2)                     # columns of one buffer
        assert not meet((at, 64, 12), (at + 12, 64, 52), 1)
        assert not meet((at, 1 << 33, 12), (at + 12, 0, 12), 1)             # one row: its stride says nothing
        assert meet((at, 1 << 33, 12), (at + (1 << 40), 4, 4), 200)


@pytest.mark.parametrize("count,elems,batch,groups,one", [
    (8, 8192, 31 * 1024, 31, False), (8, 8192, 31 * 1024 + 1, 32, True), (8, 8192, 1 << 18, 64, True),       # fewer positions than workgroups
    (3, 16384, 1 << 18, 85, True), (2, 10240, 1 << 18, 256, True), (2, 10241, 1 << 18, 128, True),           # half of the LDS
    (144, 20480, 1 << 16, 1, True), (144, 20480, (1 << 16) + 1, 1, False), (144, 20480, 1 << 18, 1, False),  # more than 128 parts: not every compute unit
    (129, 10241, 1 << 18, 1, False), (128, 20480, 1 << 17, 2, True), (128, 20480, (1 << 17) + 1, 2, False), (64, 20480, 1 << 20, 4, True),
    (144, 20480, 1, 1, False), (144, 20480, (1 << 32) - 1, 1, False), (85, 20480, (1 << 32) - 1, 3, True)])
def test_one_launch_for_table_and_positions(built, count, elems, batch, groups, one):
    # slices; parts that are whole levels take one launch for any batch
    got = ctypes.c_uint32()
    assert (bool(built.beside(count, elems, batch, 256, 1, ctypes.byref(got))), got.value) == (one, groups)
    assert built.beside(count, elems, batch, 256, 0, ctypes.byref(got)) and got.value == groups


@pytest.mark.parametrize("F", [1, 2, 4])
def test_sums_are_rounded_no_more_often_where_levels_are_spread(built, F):
    """A workgroup rounds the sum of an entry once on its way to memory: cutting by level must not put more of them on an entry than parts
    of several levels and 1024 positions to a workgroup do."""
    rng = random.Random(F)
    for _ in range(400):
        n = rng.randint(1, 16)
        sizes = [1 << rng.randint(4, 12)] * n if rng.random() < 0.6 else [rng.randint(1, 5000) for _ in range(n)]
        tables = behind_one_another(sizes)
        if rng.random() < 0.3:
            tables = [(rng.randint(0, 8000), s) for s in sizes]                    # gaps, any order, shared entries
        desc = _lib.CvPermutoDesc(dimensions=3, featureDimensionPerEntry=F, maxLevels=n, maxLevel=99.0)
        for l, (offset, size) in enumerate(tables):
            lv = desc.levelInfo[l]
            lv.currentLevelIndex, lv.offsetOfFeatureTable, lv.featureTableSize = l, offset, size
        batch = round(2 ** rng.uniform(6, 18))

        def additions(spread):
            out = (ctypes.c_uint32 * (4 * 144))()
            r = built.plan(ctypes.byref(desc), batch, 256, int(spread), out)
            assert r > 0
            parts = [tuple(out[4 * p:4 * p + 4]) for p in range(r >> 16)]
            check(parts, 0, F, tables)
            # workgroups that may add to an entry, at the first entry and in the middle of every level
            return [(r & 65535) * sum(base <= at * F < base + elems and any(o <= at < o + s for o, s in tables[first:end]) for base, elems, first, end in parts)
                    for o_, s_ in tables for at in (o_, o_ + s_ // 2)], len(parts), r & 65535
        before, parts, groups = additions(False)
        after, _, _ = additions(True)
        assert groups <= (batch - 1) // 1024 + 1
        assert all(x <= y for x, y in zip(after, before)), (F, tables, batch, before, after)
