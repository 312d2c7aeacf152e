"""planPacked (slang_amd/csrc/cv_matmul_plan.h), the host code that cuts a packed matMul call, compiled by itself: where the results lie on
the vectors, no sample's rows may be split between workgroups or leave one segment after the other."""
import ctypes
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include "cv_matmul_plan.h"
extern "C" void plan(const uint64_t* c, uint32_t* out)
{
    cv::PackedCall p = {};
    p.m = (uint32_t)c[0]; p.kt = cv::optKT((uint32_t)c[1], (uint32_t)c[9]); p.batch = (uint32_t)c[2];
    p.in = c[3]; p.inStride = c[4]; p.inBytes = c[1] * c[8]; p.out = c[5]; p.outStride = c[6]; p.outEsz = (uint32_t)c[7];
    p.fragmentBytes = (uint32_t)c[10]; p.mostPairs = (uint32_t)c[11]; p.waves = (uint32_t)c[12]; p.cus = (uint32_t)c[13];
    const cv::PackedLaunch l = cv::planPacked(p);
    out[0] = l.fits; out[1] = l.split; out[2] = l.ldsBytes; out[3] = (uint32_t)l.plan.tb; out[4] = (uint32_t)l.plan.segment; out[5] = (uint32_t)l.plan.mt;
    // every piece of a row of results: the row the kernel finds for it
    out[6] = 1;
    const uint32_t pieces = l.plan.outPieces;
    for (uint32_t i = 0; pieces && i < 16 * l.nt * pieces; ++i) out[6] &= (i * l.plan.outMagic) >> 20 == i / pieces;
}
extern "C" int overlap(const uint64_t* a, const uint64_t* b, uint32_t rows) { return cv::rowsOverlap({a[0], a[1], a[2]}, {b[0], b[1], b[2]}, rows); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(REPO, "include"),
                    "-I", os.path.join(REPO, "slang_amd", "csrc"), "-o", str(d / "plan.so"), str(d / "plan.cpp")], check=True)
    return ctypes.CDLL(str(d / "plan.so"))


# bytes of a vector's element and of a result's; k-slots, LDS bytes and most k-tiles of two tiles a fragment has; waves for up to two k-tiles
# and for more; the matrix up to which results may lie on the vectors
FLAVOURS = {"f16": (2, 2, 8, 1024, 4, 8, 8, 128), "f16to32": (2, 4, 8, 1024, 4, 8, 8, 128), "e4m3": (1, 2, 8, 512, 4, 8, 8, 128), "i8": (1, 4, 16, 1024, 4, 8, 8, 128),
            "f32": (4, 4, 8, 3072, 2, 8, 12, 64), "f32 whole": (4, 4, 8, 2048, 2, 8, 8, 64)}


def plan(lib, flavour, m, k, batch, at_in, in_stride, at_out, out_stride, cus=256):
    isz, osz, epl, fragment, pairs, few, more, _ = FLAVOURS[flavour]
    kt = -(-(-(-k // 16) * 4) // epl)
    c = (ctypes.c_uint64 * 14)(m, k, batch, at_in, in_stride, at_out, out_stride, osz, isz, epl, fragment, pairs, more if kt > 2 else few, cus)
    out = (ctypes.c_uint32 * 7)()
    lib.plan(c, out)
    return dict(zip(("fits", "split", "lds", "tb", "segment", "mt", "rows"), out))


@pytest.mark.parametrize("flavour", list(FLAVOURS))
def test_rows_on_their_vectors_stay_together(lib, flavour):
    isz, osz, most = FLAVOURS[flavour][0], FLAVOURS[flavour][1], FLAVOURS[flavour][7]
    for m in range(1, most + 1):
        for k in (1, 16, 31, 64, 65, 72, 100, most):
            if k > most:
                continue
            stride = max(m * osz, k * isz)
            for batch in (1, 17, 300, 1000, 4096, 65536, 1 << 20):
                for shift in (0, stride - m * osz):
                    p = plan(lib, flavour, m, k, batch, 4096, stride, 4096 + shift, stride)
                    assert p["fits"] and not p["split"] and p["lds"] <= 159 * 1024 and p["rows"], (m, k, batch, shift, p)


def test_rows_apart_are_split_for_few_samples(lib):
    assert plan(lib, "f16", 72, 72, 1000, 1 << 20, 144, 1 << 24, 144)["tb"] == 2        # three workgroups
    assert plan(lib, "f16", 120, 120, 1000, 1 << 20, 240, 1 << 24, 240)["tb"] == 2      # four
    # results in the gaps between the vectors of one buffer do not lie on them
    assert plan(lib, "f16", 72, 72, 1000, 1 << 20, 288, (1 << 20) + 144, 288)["tb"] == 2
    assert plan(lib, "f16", 72, 72, 1000, 1 << 20, 288, (1 << 20) + 142, 288)["tb"] == 5


@pytest.mark.parametrize("flavour", list(FLAVOURS))
def test_every_plan_fits(lib, flavour):
    for m in (1, 5, 16, 17, 64, 100, 128, 200, 256, 1000, 4096):
        for k in (1, 33, 64, 128, 200, 256):
            for batch in (1, 100, 5000, 1 << 20):
                osz = FLAVOURS[flavour][1]
                for stride in (m * osz, m * osz + 4 * osz, 1 << 27):
                    p = plan(lib, flavour, m, k, batch, 1 << 40, k * FLAVOURS[flavour][0], 1 << 20, stride)
                    assert p["fits"] and p["lds"] <= 159 * 1024 and 1 <= p["segment"] <= p["tb"] <= p["mt"] and p["rows"], (m, k, batch, stride, p)


def test_rows_overlap_by_their_bytes(lib):
    def overlap(a, b, rows):
        return bool(lib.overlap((ctypes.c_uint64 * 3)(*a), (ctypes.c_uint64 * 3)(*b), rows))
    for rows in (1, 2, 5):
        for sa, wa, sb, wb in ((8, 4, 8, 4), (8, 3, 8, 5), (8, 8, 8, 8), (8, 10, 8, 2), (6, 4, 8, 4), (0, 4, 0, 4)):
            for at in range(0, 60):
                a = {20 + r * sa + i for r in range(rows) for i in range(wa)}
                b = {at + r * sb + i for r in range(rows) for i in range(wb)}
                got = overlap((20, sa, wa), (at, sb, wb), rows)
                assert got or not a & b, (rows, sa, wa, sb, wb, at)
                if sa == sb and sa >= max(wa, wb) and rows > 1:      # rows at one distance: exactly, but for one region's end in the other's first gap
                    whole = {20 + r * sa + i for r in range(-9, 10) for i in range(wa)}
                    inside = not (at + (rows - 1) * sb + wb <= 20 or 20 + (rows - 1) * sa + wa <= at)
                    assert got == (inside and bool(b & whole)), (rows, sa, wa, sb, wb, at)
