// cv_permuto_parts.h -- how the table gradient of the permutohedral encoder is cut into parts for permutoTableGradKernel.
// Host code without HIP, so that it can be checked for every table without a GPU.
#pragma once
#include <cstdint>

#include "coopvec.h"
#include "cv_rows.h"

namespace cv {
namespace {

constexpr int kMaxTableParts = 144;      // with the encoder's description within 4 KB of kernel arguments
struct TablePart { uint32_t base, elems, first, end; };
struct TableParts {
    TablePart part[kMaxTableParts];
    uint32_t count, groups;          // parts, and workgroups to a part
    uint32_t sliced;                 // some part is a slice of a level's entries
};

// The doubles that half and the whole of a compute unit's LDS (160 KB) hold.
constexpr uint64_t kPartHalf = 80 * 1024 / 8, kPartMost = 160 * 1024 / 8;

// Cuts the table into parts for permutoTableGradKernel: consecutive levels as long as the range from the first to the last of
// their entries fits half of a compute unit's LDS, so that two workgroups of 16 waves share it; a level beyond that by itself,
// up to the whole 160 KB; and a level beyond those in slices of its entries, each walked by all positions of the batch.  A slice
// repeats the search for the simplex: 2^18 positions on 8 levels of 2^16 two-feature entries, seven slices each, take 128 us, on
// levels of 2^17 in thirteen slices 219 us, and either takes 6.3 to 6.7 ms with the additions in memory.  Sixteen slices at most,
// since the list of parts travels with the kernel's arguments.
// Levels may lie anywhere: with gaps between them (a sum that stays zero is not added to memory), in any order, on the same
// entries (each part adds its sums to memory atomically).
// False: more parts than that, or elements whose numbers exceed 32 bits.
inline bool cutTable(const CvPermutoDesc& desc, TableParts& t, uint64_t together = kPartHalf)
{
    const uint64_t F = (uint64_t)desc.featureDimensionPerEntry;
    t.count = 0;
    t.sliced = 0;
    bool whole = false;      // the part before this level is made of whole levels
    // (together: the most elements that levels share a part up to)
    for (uint32_t l = 0; l < desc.maxLevels; ++l) {
        const CvPermutoLevelInfo& lv = desc.levelInfo[l];
        const uint64_t from = (uint64_t)lv.offsetOfFeatureTable * F, elems = (uint64_t)lv.featureTableSize * F, to = from + elems;
        if (to > 0xffffffffull) return false;
        if (whole) {
            TablePart& last = t.part[t.count - 1];
            const uint64_t lastTo = (uint64_t)last.base + last.elems;
            const uint64_t lo = from < last.base ? from : last.base, hi = to > lastTo ? to : lastTo;
            if (hi - lo <= together) {
                last.base = (uint32_t)lo;
                last.elems = (uint32_t)(hi - lo);
                last.end = l + 1;
                continue;
            }
        }
        // whole entries to a slice: as many slices as their number needs, so that none comes out above kPartMost
        const uint64_t entries = lv.featureTableSize, most = kPartMost / F, slices = (entries + most - 1) / most;
        if (slices == 0 || slices > 16) return false;
        if (slices > 1) t.sliced = 1;
        whole = slices == 1;
        const uint64_t perSlice = (entries + slices - 1) / slices * F;
        for (uint64_t at = 0; at < elems; at += perSlice) {
            if (t.count == (uint32_t)kMaxTableParts) return false;
            t.part[t.count++] = TablePart{(uint32_t)(from + at), (uint32_t)(elems - at < perSlice ? elems - at : perSlice), l, l + 1};
        }
    }
    return t.count > 0;
}

// As many workgroups (of 1024 threads) as the compute units hold, dealt evenly to the parts, and none without 1024 positions.
inline uint32_t largestPart(const TableParts& t)
{
    uint32_t most = 0;
    for (uint32_t p = 0; p < t.count; ++p) most = t.part[p].elems > most ? t.part[p].elems : most;
    return most;
}
inline void dealGroups(TableParts& t, uint32_t batch, uint32_t cus)
{
    const uint32_t resident = cus * (largestPart(t) <= kPartHalf ? 2u : 1u), want = (batch - 1u) / 1024u + 1u;
    const uint32_t each = resident / t.count ? resident / t.count : 1u;
    t.groups = want < each ? want : each;
}

// One level to a part instead of several where the parts leave compute units without a workgroup of 1024 positions: a level's additions in LDS, not
// its start, are what a workgroup takes its time for.  Several levels to a part against one (and position gradients beside), 3 dimensions, us: 6 levels of
// 2^9 four-feature entries over 4096 / 2^14 / 2^16 positions 48.5, 48.5, 49.1 against 14.1, 14.4, 21.1; 8 levels of 2^10 two-feature entries over 20000
// / 2^16 30.8, 31.9 against 8.9, 12.7; 2 dimensions, 8 levels of 2^8 of two over 20000 / 2^16 / 2^17 (one part) 19.7, 20.4, 21.9 against 7.1, 9.5,
// 14.6, and over 2^18 25.1 against 28.3.  (Below kFewPositions there is little to spread.)
// Each workgroup of a part rounds its sums to float once, on their way to memory.  A part of one level has no more workgroups than the part of several it
// came from, so no entry's sum is rounded more often; levels on the same entries, whose addends one part sums in double, stay together.  (Fewer
// positions to a workgroup, 512 or 256, would halve the time over 4096 positions, 6 levels of 2^9 four-feature entries 14.1 -> 6.9 us, but put the gradient
// 8.3e-8 of its norm off the 64-bit one instead of 5.3e-8.)
constexpr uint32_t kFewPositions = 2048u;
inline bool levelsApart(const CvPermutoDesc& desc)
{
    for (uint32_t l = 0; l < desc.maxLevels; ++l)
        for (uint32_t m = 0; m < l; ++m) {
            const CvPermutoLevelInfo &a = desc.levelInfo[l], &b = desc.levelInfo[m];
            if ((uint64_t)a.offsetOfFeatureTable < (uint64_t)b.offsetOfFeatureTable + b.featureTableSize &&
                (uint64_t)b.offsetOfFeatureTable < (uint64_t)a.offsetOfFeatureTable + a.featureTableSize) return false;
        }
    return true;
}
inline bool cutByLevel(const CvPermutoDesc& desc, uint32_t batch, uint32_t cus, TableParts& t)
{
    if (t.sliced || t.count >= desc.maxLevels || batch < kFewPositions || (uint64_t)t.count * ((batch - 1u) / 1024u + 1u) >= cus || !levelsApart(desc)) return false;
    return cutTable(desc, t, 0);      // (levels that were joined are whole ones, no more than a description has)
}

// The parts and workgroups of a launch; spread: cutByLevel may be asked (entries of 1, 2 or 4 features, position gradients that do not lie on what
// is read).  False: no parts.
inline bool planTable(const CvPermutoDesc& desc, uint32_t batch, uint32_t cus, bool spread, TableParts& t)
{
    if (!cutTable(desc, t)) return false;
    if (spread) cutByLevel(desc, batch, cus, t);
    dealGroups(t, batch, cus);
    return true;
}

// Whether position gradients go into the table's launch (of several parts; after dealGroups).  Always where parts are whole levels; two launches against one,
// us: 3 dimensions, 8 levels of 2^12 two-feature entries over 65 / 1024 / 4096 / 2^14 positions 11.1, 16.6, 17.2, 19.4 against 8.9, 10.0, 9.5, 9.7; 5 levels of
// 2^11 three-feature ones over 65 / 4096 / 24000 18.8, 28.1, 28.2 against 14.9, 16.5, 16.9; 2 levels of 2^12 over 65 / 30000 6.9, 12.8 against 5.2, 10.1; 4
// dimensions, 8 levels of 2^9 four-feature entries over one position 17.4 against 12.2.
// Slices: not with too few positions for workgroups on every compute unit: spread by a kernel of their own they are done sooner.  And not where a part has but
// one or two workgroups and many positions: a table of 91 parts or more, whose grid leaves compute units without one or deals some of them twice the
// work.  One launch against two, 3 dimensions, 9 or 7 levels of two-feature entries, 2^14 / 2^16 / 2^18 positions: 144 parts (144
// workgroups) 41.7, 149, 606 us against 53.9, 150, 542; 126 parts (252) 24.0, 79.2, 304 against 36.6, 86.5, 288; 105 parts (210) 23.7,
// 77.2, 297 against 33.2, 81.7, 276; 64 parts (256) 62.5 and 258 against 84.6 and 273 over 2^16 and 2^18, and still 1063 against 1108 over 2^20.
inline bool positionsBeside(const TableParts& t, uint32_t batch, uint32_t cus)
{
    return !t.sliced || ((uint64_t)t.count * ((batch - 1u) / 1024u + 1u) >= cus && !(t.groups <= 2u && batch > 65536u * t.groups));
}

} // namespace
} // namespace cv
