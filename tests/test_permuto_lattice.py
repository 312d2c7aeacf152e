"""LatticeSimplex and LatticeSimplexAny (slang_amd/csrc/cv_permuto_lattice.h), compiled for the host and compared with the
lattice steps as the reference writes them (permuto-encoder.slang:74-179, :296-309: ranks counted, arrays indexed by rank,
keys hashed one by one): weights and hashes bit for bit, the gradients of the elevated coordinates too.  Every number of
dimensions, positions at random, on the coarse grids where coordinates tie and elevated values lie half way between lattice
points, at the end of LatticeSimplex's reach and beyond it (LatticeSimplexAny alone)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from slang_amd import _lib

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include <cmath>
#include "cv_permuto_lattice.h"
using namespace cv;

// false: rounding far out leaves ranks beyond 0..D, for which the reference has no answer
template <int D> static bool reference(const float* pos, const CvPermutoLevelInfo& lv, const float* dbary, float* bary, uint32_t* hash, float* delev)
{
    float elevated[D + 1], sum = 0.0f;
    for (int dim = D - 1; dim >= 0; --dim) {
        const float cf = (pos[dim] + lv.shiftsPerDim[dim]) * lv.scalesPerDim[dim];
        elevated[dim + 1] = sum - (float)(dim + 1) * cf;
        sum += cf;
    }
    elevated[0] = sum;
    int rem0[D + 1], rank[D + 1], isum = 0;
    for (int dim = 0; dim <= D; ++dim) {
        rank[dim] = 0;
        const float v = elevated[dim] * (1.0f / (float)(D + 1));
        const float up = ceilf(v) * (float)(D + 1), down = floorf(v) * (float)(D + 1);
        rem0[dim] = (up - elevated[dim] < elevated[dim] - down) ? (int)up : (int)down;
        isum += rem0[dim];
    }
    isum /= (D + 1);
    for (int dim = 0; dim < D; ++dim)
        for (int other = dim + 1; other <= D; ++other) {
            if (elevated[dim] - (float)rem0[dim] < elevated[other] - (float)rem0[other]) rank[dim]++;
            else rank[other]++;
        }
    for (int dim = 0; dim <= D; ++dim) {
        rank[dim] += isum;
        if (rank[dim] < 0) { rank[dim] += D + 1; rem0[dim] += D + 1; }
        else if (rank[dim] > D) { rank[dim] -= D + 1; rem0[dim] -= D + 1; }
    }
    for (int dim = 0; dim <= D; ++dim)
        if (rank[dim] < 0 || rank[dim] > D) return false;
    float b[D + 2] = {};
    for (int dim = 0; dim <= D; ++dim) {
        const float delta = (elevated[dim] - (float)rem0[dim]) * (1.0f / (float)(D + 1));
        b[D - rank[dim]] += delta;
        b[D + 1 - rank[dim]] -= delta;
    }
    b[0] += 1.0f + b[D + 1];
    float db[D + 2];
    for (int k = 0; k <= D; ++k) { bary[k] = b[k]; db[k] = dbary[k]; }
    db[D + 1] = db[0];
    for (int dim = 0; dim <= D; ++dim) delev[dim] = (db[D - rank[dim]] - db[D + 1 - rank[dim]]) * (1.0f / (float)(D + 1));
    for (int k = 0; k <= D; ++k) {
        uint32_t h = 0;
        for (int dim = 0; dim < D; ++dim) {
            int key = rem0[dim] + k;
            if (rank[dim] > D - k) key -= D + 1;
            h += (uint32_t)key;
            h *= 2531011u;
        }
        hash[k] = h;
    }
    return true;
}

static long differ(float a, float b) { return !(a == b || (a != a && b != b)); }     // (signed zeros are one value)

template <int D, typename Simplex> static long differences(const float* pos, const float* db, const CvPermutoLevelInfo& lv, uint32_t hashBits)
{
    float b[D + 1], de[D + 1], got[D + 1], dbary[D + 1];
    uint32_t h[D + 1];
    for (int k = 0; k <= D; ++k) dbary[k] = db[k];
    if (!reference<D>(pos, lv, dbary, b, h, de)) return 0;
    Simplex s;
    s.search(pos, latticeLevel<D>(lv));
    s.toElevated(dbary, got);
    long off = 0;
    for (int k = 0; k <= D; ++k) off += differ(b[k], s.bary[k]) + (((h[k] ^ s.hash[k]) & hashBits) != 0u) + differ(de[k], got[k]);
    return off;
}

template <int D> static long compare(const float* pos, const float* db, long n, const CvPermutoDesc& desc, long* within)
{
    const float reach = latticeReach(desc);
    long bad = 0;
    for (long i = 0; i < n; ++i, pos += D, db += D + 1) {
        bad += differences<D, LatticeSimplexAny<D>>(pos, db, desc.levelInfo[0], 0xffffffffu) != 0;
        if constexpr (D <= 4) {
            bool in = true;
            for (int d = 0; d < D; ++d) in = in && fabsf(pos[d]) <= reach;
            *within += in;
            if (in) bad += differences<D, LatticeSimplex<D>>(pos, db, desc.levelInfo[0], 0xffffffu) != 0;
        }
    }
    return bad;
}

extern "C" long check(int D, const float* pos, const float* dbary, long n, const CvPermutoDesc* d, long* within)
{
    switch (D) {
    case 1: return compare<1>(pos, dbary, n, *d, within);
    case 2: return compare<2>(pos, dbary, n, *d, within);
    case 3: return compare<3>(pos, dbary, n, *d, within);
    case 4: return compare<4>(pos, dbary, n, *d, within);
    case 5: return compare<5>(pos, dbary, n, *d, within);
    case 6: return compare<6>(pos, dbary, n, *d, within);
    case 7: return compare<7>(pos, dbary, n, *d, within);
    case 8: return compare<8>(pos, dbary, n, *d, within);
    }
    return -1;
}
"""


@pytest.fixture(scope="module")
def lattice(tmp_path_factory):
    d = tmp_path_factory.mktemp("lattice")
    (d / "lattice.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I", os.path.join(REPO, "include"),
                    "-I", os.path.join(REPO, "slang_amd", "csrc"), "-o", str(d / "lattice.so"), str(d / "lattice.cpp")], check=True)
    lib = ctypes.CDLL(str(d / "lattice.so"))
    lib.check.restype = ctypes.c_long

    def call(D, pos, dbary, scales, shifts):
        desc = _lib.CvPermutoDesc(dimensions=D, featureDimensionPerEntry=2, maxLevels=1, maxLevel=1.0)
        for i in range(D):
            desc.levelInfo[0].scalesPerDim[i], desc.levelInfo[0].shiftsPerDim[i] = float(scales[i]), float(shifts[i])
        pos, dbary = np.ascontiguousarray(pos, np.float32), np.ascontiguousarray(dbary, np.float32)
        within = ctypes.c_long(0)
        return lib.check(D, pos.ctypes.data_as(ctypes.c_void_p), dbary.ctypes.data_as(ctypes.c_void_p), ctypes.c_long(len(pos)), ctypes.byref(desc), ctypes.byref(within)), within.value
    return call


@pytest.mark.parametrize("D", range(1, 9))
def test_simplex_equals_the_steps_of_the_reference(lattice, D):
    rng = np.random.default_rng(D)
    n = 20000
    own = [1.0 / np.sqrt((d + 1) * (d + 2)) for d in range(D)]
    dbary = rng.standard_normal((n, D + 1))
    kinds = {
        "uniform": (rng.random((n, D)), [4.0 * s for s in own], rng.uniform(-5, 5, D)),
        "fine level": (rng.random((n, D)), [512.0 * s for s in own], rng.uniform(-5, 5, D)),
        "wide": (rng.uniform(-300, 300, (n, D)), [16.0 * s for s in own], rng.uniform(-5, 5, D)),
        "ties": (rng.integers(-8, 9, (n, D)), [1.0] * D, [0.0] * D),
        "half way": (rng.integers(-64, 65, (n, D)) / 4.0, [0.5] * D, [0.0] * D),
        "half way, shifted": (rng.integers(-64, 65, (n, D)) / 8.0, [(D + 1) / 2.0] * D, [0.125] * D),
        "one ulp off half way": (np.nextafter(np.float32(rng.integers(-16, 17, (n, D)) / 2.0), np.float32(rng.choice([-1, 1], (n, D)) * 1e9)), [1.0] * D, [0.0] * D),
        "end of the reach": (rng.uniform(-1, 1, (n, D)) * 2.0 ** 20, [2.0 / (D + 1) ** 2] * D, rng.uniform(-5, 5, D)),
        "beyond the reach": (rng.uniform(-1, 1, (n, D)) * 2.0 ** 26, [1.0] * D, rng.uniform(-5, 5, D)),
    }
    # (an elevated value below 2^-147, one ulp off zero, is zero after the division by D + 1)
    kinds["one ulp off half way"][0][np.abs(kinds["one ulp off half way"][0]) < 1e-30] = 0.5
    for name, (pos, scales, shifts) in kinds.items():
        bad, within = lattice(D, pos, dbary, scales, shifts)
        assert bad == 0, name
        if D <= 4:
            assert (within > 0.9 * n) == (name != "beyond the reach"), (name, within)
