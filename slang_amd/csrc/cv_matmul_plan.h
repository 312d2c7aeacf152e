// cv_matmul_plan.h -- how the packed matMul (cv_matmul_packed.h) cuts a call: row tiles to a workgroup, results that wait in LDS together,
// tiles and waves.  Without HIP, so that it can be checked for every call without a GPU.
#pragma once
#include "cv_layout.h"
#include "cv_rows.h"

namespace cv {

constexpr uint32_t kPackedLds = 159u * 1024u;      // (__syncthreads_or has some of its own)

// the kernel's argument
struct PackedPlan {
    int32_t mt, tb;                  // row tiles of the matrix, of a workgroup's block (blockIdx.y)
    int32_t segment;                 // row tiles whose results wait in LDS together
    uint32_t outRow;                 // bytes from one sample's results to the next in LDS
    uint32_t stageBytes;             // a wave's part of the LDS
    uint32_t outPieces, outMagic;    // 16-byte pieces of a row of results (a segment) and 2^20 / outPieces, rounded up; 0: one block
    int32_t outElements;             // the results leave element by element
    int32_t outLines;                // rows and segments of results are whole 128-byte lines: they pass by the caches (storeStream16)
    uint64_t matBytes;               // RowMajor matrices at least a lane-chunk long: their bytes, else 0
};

// a call: vectors, results, and what a flavour's matrix takes
struct PackedCall {
    uint32_t m, kt, batch;
    uint64_t in, inStride, inBytes, out, outStride;      // (addresses; inBytes: of a vector)
    uint32_t outEsz;                 // bytes of a result
    uint32_t fragmentBytes;          // of LDS to a fragment
    uint32_t mostPairs;              // k-tiles up to which a wave takes two tiles (registers)
    uint32_t waves;                  // to a workgroup
    bool accumulate;
    uint32_t cus;
};

struct PackedLaunch {
    PackedPlan plan;
    uint32_t ldsBytes, nt;           // 16-sample tiles of a wave
    bool fits, split;                // split: the rows of a sample's results come from several workgroups, or leave a segment after the other
};

// How rows of `bytes` bytes leave: as one block (pieces = 0) where they lie one behind the other, or in pieces of every row.  False: rows
// shorter than a piece that are not packed.
inline bool rowsInPieces(uint64_t base, uint64_t stride, uint32_t bytes, PackedPlan& p)
{
    p.outPieces = p.outMagic = 0u;
    p.outRow = bytes % 16u ? bytes : bytes + 16u;      // (so that the 16 rows of a tile lie on different banks)
    if ((base & 15u) == 0 && stride == bytes && bytes % 16u) return true;
    if (bytes < 16u || stride >= (1u << 26)) return false;
    p.outPieces = (bytes + 15u) / 16u;
    p.outMagic = ((1u << 20) + p.outPieces - 1u) / p.outPieces;
    return true;
}

inline PackedLaunch planPacked(const PackedCall& c)
{
    PackedLaunch l = {};
    PackedPlan& p = l.plan;
    const uint32_t mt = optMT(c.m), rowBytes = c.m * c.outEsz;
    p.mt = (int32_t)mt;
    l.nt = c.kt <= c.mostPairs && c.batch / 32u >= c.cus * 8u ? 2u : 1u;
    auto plan = [&](uint32_t blocks, uint32_t nt, uint32_t mostStage) {
        l.nt = nt;
        p.tb = (int32_t)((mt + blocks - 1) / blocks);
        const uint32_t tileBytes = 16u * nt * 16u * c.outEsz;
        p.outElements = c.accumulate;
        p.segment = p.tb;
        if (blocks == 1 && mt * tileBytes <= mostStage) {
            if (!rowsInPieces(c.out, c.outStride, rowBytes, p)) p.outElements = 1;
        } else {
            const int most = (int)(mostStage / tileBytes);
            if (most < p.tb) p.segment = most;
            p.outPieces = (uint32_t)p.segment * c.outEsz;
            p.outRow = 16u * p.outPieces + 16u;
            p.outMagic = ((1u << 20) + p.outPieces - 1u) / p.outPieces;
            if (c.outStride >= (1u << 26)) p.outElements = 1;
        }
        p.stageBytes = (16u * nt * p.outRow + 15u) / 16u * 16u;
        l.ldsBytes = (uint32_t)p.tb * (c.kt * c.fragmentBytes + 64u) + c.waves * p.stageBytes;
        l.fits = l.ldsBytes <= kPackedLds;
        l.split = p.tb < p.mt || p.segment < p.tb;
        const uint32_t segmentBytes = p.segment == (int32_t)mt ? rowBytes : (uint32_t)p.segment * 16u * c.outEsz;
        p.outLines = ((c.out | c.outStride | rowBytes | segmentBytes) & 127u) == 0;
    };
    const uint32_t wanted = l.nt;
    // Results on top of the vectors: a wave reads all that it needs of a sample before it stores the first of its results, and nobody else
    // reads that sample.
    if (rowsOverlap(Rows{c.in, c.inStride, c.inBytes}, Rows{c.out, c.outStride, rowBytes}, c.batch)) {
        for (uint32_t n = wanted; n >= 1; --n) {
            plan(1u, n, kPackedLds);
            if (l.fits) return l;
        }
    }
    // a batch that leaves compute units idle: the rows are split between them, down to a lane-chunk of the matrix a thread
    const uint32_t groups = (uint32_t)(((uint64_t)c.batch + 16 * wanted * c.waves - 1) / (16 * wanted * c.waves));
    uint32_t blocks = 1;
    while (blocks < mt && groups * (blocks + 1) <= c.cus && (mt + blocks - 1) / blocks * c.kt > 8u) ++blocks;
    // where the LDS is short, fewer results wait, then a wave takes one tile, then the rows are split
    l.fits = false;
    for (; !l.fits && blocks <= mt; ++blocks)
        for (uint32_t n = wanted; !l.fits && n >= 1; --n)
            for (uint32_t stage = 8192u; !l.fits && stage >= 2048u; stage /= 2u) plan(blocks, n, stage);
    return l;
}

} // namespace cv
