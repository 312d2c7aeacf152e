// cv_permuto_impl.h -- one level of PermutoEncoder::encode (source/standard-modules/neural/permuto-encoder.slang:240-337) for one
// position, shared by the encoder kernels: the simplex (cv_permuto_lattice.h), its vertices' slots of the hashed feature table
// (:296-309) and their entries weighted.  Line numbers in the comments below refer to that file.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "coopvec.h"
#include "cv_permuto_lattice.h"

namespace cv {

// Slot of a vertex with this hash in the feature table of its level (:305-309), in entries.  A table of 2^n entries, which is
// what prepareLevelInfo makes, is indexed with a mask: the general remainder is a division by a run-time value, some forty
// instructions per vertex.  PLAIN (permutoPlainLevels): every table has 2^n entries, n <= 24.  Then no lane needs the remainder,
// whose branch cost four divergent regions per level and kept the loads of the vertices apart.
template <bool PLAIN>
__device__ __forceinline__ uint32_t vertexSlot(uint32_t size, uint32_t hash)
{
    return PLAIN || (size & (size - 1u)) == 0u ? (hash & (size - 1u)) : hash % size;
}

// Some lane's position lies beyond what LatticeSimplex takes (or is not a number): the wave takes LatticeSimplexAny.
template <int D>
__device__ __forceinline__ bool anyBeyondReach(const float* pos, float reach)
{
    bool beyond = false;
#pragma unroll
    for (int d = 0; d < D; ++d) beyond = beyond | !(__builtin_fabsf(pos[d]) <= reach);
    return __any(beyond);
}

// Every level has a table of 2^n entries, n <= 24, and none lies beyond maxLevel: what an encoder prepared by the library
// and used with all its levels has.  (A table of no entries is not plain.)
inline bool permutoPlainLevels(const CvPermutoDesc& desc)
{
    for (uint32_t l = 0; l < desc.maxLevels; ++l) {
        const CvPermutoLevelInfo& lv = desc.levelInfo[l];
        const uint32_t size = lv.featureTableSize;
        if (size == 0u || size > (1u << 24) || (size & (size - 1u)) != 0u || (float)lv.currentLevelIndex >= desc.maxLevel + 1e-3f) return false;
    }
    return true;
}

// F consecutive elements of type T: one entry of the feature table, one level's share of an encoded vector
template <typename T, int F>
struct PermutoEntry { typedef T type __attribute__((ext_vector_type(F))); };

// One level of encode for one position (:259-317): zeros beyond maxLevel, else the entries of the simplex vertices
// weighted in T, vertex by vertex.  `table` may point to memory or to a copy of the table in LDS; entries are read
// whole, so `table` and every entry offset must be multiples of the entry size.
// PLAIN: a level of an encoder that permutoPlainLevels accepts.  Simplex: LatticeSimplexAny<D>, or LatticeSimplex<D> if PLAIN
// and no lane is beyond its reach.
template <typename T, int D, int F, bool PLAIN, typename Simplex>
__device__ __forceinline__ typename PermutoEntry<T, F>::type permutoEncodeEntry(const float* pos, const LatticeLevel<D>& lv, const T* table, float maxLevel)
{
    typedef typename PermutoEntry<T, F>::type Entry;
    Entry acc;
#pragma unroll
    for (int f = 0; f < F; ++f) acc[f] = (T)0.f;
    if (PLAIN || !((float)lv.index >= maxLevel + 1e-3f)) {   // zero padding beyond maxLevel, :259-262
        Simplex simplex;
        simplex.search(pos, lv);
        const Entry* entries = (const Entry*)table + lv.offset;
        Entry e[D + 1];
#pragma unroll
        for (int k = 0; k <= D; ++k) e[k] = entries[vertexSlot<PLAIN>(lv.size, simplex.hash[k])];
        T w[D + 2];                                          // in pairs: one conversion for two halves
#pragma unroll
        for (int k = 0; k <= D; k += 2) {
            typedef T Pair __attribute__((ext_vector_type(2)));
            typedef float FloatPair __attribute__((ext_vector_type(2)));
            const Pair p = __builtin_convertvector((FloatPair{simplex.bary[k], simplex.bary[k < D ? k + 1 : k]}), Pair);
            w[k] = p.x; w[k + 1] = p.y;
        }
#pragma unroll
        for (int k = 0; k <= D; ++k)
#pragma unroll
            for (int f = 0; f < F; ++f) acc[f] = (T)(acc[f] + (T)(w[k] * e[k][f]));    // in T, vertex by vertex (:312-316)
    }
    return acc;
}

} // namespace cv
