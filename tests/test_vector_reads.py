"""Where the kernels read vectors of any length (slang_amd/csrc/cv_reads.h), compiled by itself: for every size, lane group and
fragment, no read may touch a byte outside the batch's vectors, and every element of a lane's slice must come out at its place.

The loops below make the reads of the three kernels that take such vectors: equal-layer forward (mlpForwardKernel, load mode 1),
chain forward (mlpChainKernel without QUAD) and packed matMul (packedRows)."""
import ctypes
import os
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include <vector>
#include "cv_reads.h"
using namespace cv;
namespace {
uint64_t faults, end;
std::vector<uint8_t> memory;
// `bytes` bytes at `at`, moved down by `down`, into x (whose other bytes stay)
void read(uint64_t at, uint32_t bytes, uint32_t down, uint8_t* x)
{
    if (at + bytes > end || at > end) { ++faults; return; }
    for (uint32_t b = 0; b + down < bytes; ++b) x[b] = memory[at + b + down];
}
// the first `valid` bytes of x must be those at `want`
void expect(const uint8_t* x, uint64_t want, int valid, int most)
{
    for (int b = 0; b < valid && b < most; ++b)
        if (want + b >= end || x[b] != memory[want + b]) ++faults;
}
void start(uint32_t batch, uint64_t stride, uint32_t in, uint32_t esz)
{
    faults = 0;
    end = vectorsEnd(batch, stride, in, esz);
    memory.resize(end);
    uint32_t v = 12345u;
    for (uint8_t& b : memory) { v = v * 1664525u + 1013904223u; b = (uint8_t)(v >> 24); }
}
uint64_t least(uint64_t a, uint64_t b) { return a < b ? a : b; }
// loadUpTo (cv_stage.h): a fragment of `dwords` dwords
void readUpTo(uint64_t want, uint32_t dwords, uint8_t* x)
{
    const uint32_t part = dwords % 4 == 0 ? 16 : 8;
    for (uint32_t d = 0; d < 4 * dwords; d += part) {
        read(readAt(want + d, part, end), part, readDown(want + d, part, end), x + d);
    }
}
}

// super-tiles of `samples` vectors
extern "C" uint64_t equalLayers(uint32_t in, uint32_t esz, uint32_t batch, uint64_t stride, uint32_t samples)
{
    start(batch, stride, in, esz);
    if (end < 16) return 0;
    const uint32_t gs = optGS(in), KT = optKT(in, 8);
    for (uint64_t t = 0; t * samples < batch + samples; ++t) {      // (one beyond the batch: a wave without a tile)
        const bool inside = tileReadsEnd(t * samples, samples, stride, gs, 8 * KT, esz) <= end;
        for (uint32_t i = 0; i < samples; ++i)
            for (uint32_t g = 0; g < 4; ++g)
                for (uint32_t kt = 0; kt < KT; ++kt) {
                    const int valid = sliceBytes(in, gs, g, esz);
                    const uint32_t bytes = kt + 1 == KT && gs <= 8 * KT - 4 ? 4 * esz : 8 * esz;
                    const uint64_t s = inside ? t * samples + i : least(t * samples + i, batch - 1);
                    const uint64_t want = s * stride + (valid > 0 ? g * gs * esz : 0) + kt * 8 * esz;
                    uint8_t x[16] = {};
                    if (inside) read(want, bytes, 0, x);
                    else read(readAt(want, bytes, end), bytes, readDown(want, bytes, end), x);
                    expect(x, want, valid - (int)(kt * 8 * esz), (int)bytes);
                }
    }
    return faults;
}

// tiles of `samples` vectors, `slots` k-slots to a fragment; tail: dwords of the last fragment that are read inside (0: all)
static uint64_t wholeReads(uint32_t in, uint32_t esz, uint32_t batch, uint64_t stride, uint32_t samples, uint32_t slots, bool chain)
{
    start(batch, stride, in, esz);
    if (end < 16) return 0;
    const uint32_t gs = optGS(in), KT = optKT(in, slots), dwords = slots * esz / 4;
    const uint32_t rest = gs - (KT - 1) * slots;      // k-slots of the last fragment
    const uint32_t tail = chain ? (rest <= 4 ? esz * 4 : slots * esz) : (rest * esz == 12 ? 16 : rest * esz);
    for (uint64_t t = 0; t * samples < batch; ++t) {
        const bool inside = tileReadsEnd(t * samples, samples, stride, gs, slots * KT, esz) <= end;
        for (uint32_t i = 0; i < samples; ++i)
            for (uint32_t g = 0; g < 4; ++g)
                for (uint32_t kt = 0; kt < KT; ++kt) {
                    const int valid = sliceBytes(in, gs, g, esz) - (int)(kt * slots * esz);
                    const uint64_t s = inside ? t * samples + i : least(t * samples + i, batch - 1);
                    const uint64_t want = s * stride + g * gs * esz + kt * slots * esz;
                    uint8_t x[32] = {};
                    if (inside) read(want, kt + 1 == KT ? tail : 4 * dwords, 0, x);
                    else readUpTo(want, dwords, x);
                    expect(x, want, valid, 4 * (int)dwords);
                }
    }
    return faults;
}
extern "C" uint64_t chain(uint32_t in, uint32_t esz, uint32_t batch, uint64_t stride) { return wholeReads(in, esz, batch, stride, 16, 8, true); }
extern "C" uint64_t packed(uint32_t in, uint32_t esz, uint32_t batch, uint64_t stride, uint32_t samples, uint32_t slots) { return wholeReads(in, esz, batch, stride, samples, slots, false); }
"""


@pytest.fixture(scope="module")
def reads(tmp_path_factory):
    d = tmp_path_factory.mktemp("reads")
    (d / "reads.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(REPO, "include"),
                    "-I", os.path.join(REPO, "slang_amd", "csrc"), "-o", str(d / "reads.so"), str(d / "reads.cpp")], check=True)
    lib = ctypes.CDLL(str(d / "reads.so"))
    u32, u64 = ctypes.c_uint32, ctypes.c_uint64
    for name, args in (("equalLayers", [u32, u32, u32, u64, u32]), ("chain", [u32, u32, u32, u64]), ("packed", [u32, u32, u32, u64, u32, u32])):
        getattr(lib, name).argtypes, getattr(lib, name).restype = args, u64
    return lib


BATCHES = list(range(1, 19)) + [31, 32, 33, 63, 64, 65, 79, 127, 128, 129, 200]
PADS = (0, 1, 3, 40)      # elements between one vector and the next


@pytest.mark.parametrize("esz", [1, 2])
def test_equal_layer_reads_stay_in_the_vectors(reads, esz):
    bad = [(size, batch, pad, samples) for size in range(1, 65) for batch in BATCHES for pad in PADS for samples in (32, 64, 128)
           if reads.equalLayers(size, esz, batch, (size + pad) * esz, samples)]
    assert not bad, (sorted({b[0] for b in bad}), bad[:4])


@pytest.mark.parametrize("esz", [1, 2, 4])
def test_chain_reads_stay_in_the_vectors(reads, esz):
    bad = [(size, batch, pad) for size in range(1, 129) for batch in BATCHES for pad in PADS if reads.chain(size, esz, batch, (size + pad) * esz)]
    assert not bad, (sorted({b[0] for b in bad}), bad[:4])


@pytest.mark.parametrize("esz,slots,most", [(1, 8, 256), (1, 16, 256), (2, 8, 256), (4, 8, 256)])
def test_packed_reads_stay_in_the_vectors(reads, esz, slots, most):
    bad = [(size, batch, pad, samples) for size in range(1, most + 1) for batch in BATCHES for pad in PADS for samples in (16, 32)
           if reads.packed(size, esz, batch, (size + pad) * esz, samples, slots)]
    assert not bad, (sorted({b[0] for b in bad}), bad[:4])


def test_a_read_that_begins_behind_the_end(reads):
    # a lane's second fragment behind the last vector (50 halves, lane group 3: its slice ends at element 50, the fragment begins at 56)
    assert reads.equalLayers(50, 2, 1, 100, 32) == 0
