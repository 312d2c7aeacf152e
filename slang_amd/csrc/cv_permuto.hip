// cv_permuto.hip -- input encoders of the neural module in front of the MLP, for gfx950.
//
// Replaces, for a whole batch of positions, PermutoEncoder::encode and its reverse mode
// (source/standard-modules/neural/permuto-encoder.slang:240-337, readFeatureValueBwd :222-238,
// prepareLevelInfo :339-368) and the grid hashes it is built on
// (source/standard-modules/neural/hash-function.slang:69-151).  A thread handles one position and level (or all levels of a
// position, one after the other): it finds the enclosing simplex of the permutohedral lattice and gathers D+1 hashed
// feature-table entries.  With the table in LDS the arithmetic binds: 160 to 230 vector instructions per position and
// level in two and three dimensions kept the vector-ALU port full, some 130 in three do now (LatticeSimplex).  The reverse pass adds every position's contributions to the
// table gradient up in LDS, by parts of the table, and only the sums to memory; tables that cannot be cut so, and a handful of
// positions, are added in memory with atomics, as the reference does.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>

#include "cv_device.h"
#include "cv_error.h"
#include "cv_kernels.h"
#include "cv_launch.h"
#include "cv_permuto_impl.h"
#include "cv_permuto_parts.h"

namespace cv {
namespace {

constexpr int kMaxDims = CV_PERMUTO_MAX_DIMS;
constexpr int kMaxLevels = CV_PERMUTO_MAX_LEVELS;

// ---- hashes (hash-function.slang) -----------------------------------------------------------
struct Pcg32 {
    uint64_t state, inc;
    __host__ __device__ uint32_t next()                               // :35-42
    {
        const uint64_t old = state;
        state = old * 0x5851f42d4c957f2dULL + inc;
        const uint32_t xorshifted = (uint32_t)(((old >> 18) ^ old) >> 27);
        const uint32_t rot = (uint32_t)(old >> 59);
        return (xorshifted >> rot) | (xorshifted << ((~rot + 1u) & 31u));
    }
    __host__ __device__ void init(uint64_t initstate, uint64_t initseq = 1)   // :25-32
    {
        state = 0;
        inc = (initseq << 1) | 1u;
        next();
        state += initstate;
        next();
    }
    __host__ __device__ void advance(int64_t delta)                    // :45-65
    {
        uint64_t curMult = 0x5851f42d4c957f2dULL, curPlus = inc, accMult = 1, accPlus = 0;
        for (uint64_t d = (uint64_t)delta; d > 0; d /= 2) {
            if (d & 1) { accMult *= curMult; accPlus = accPlus * curMult + curPlus; }
            curPlus = (curMult + 1) * curPlus;
            curMult *= curMult;
        }
        state = accMult * state + accPlus;
    }
};

__host__ __device__ inline uint32_t baseConvertHash(const uint32_t* pos, int dims)   // :103-113
{
    uint32_t k = 0;
    for (int d = 0; d < dims; ++d) { k += pos[d]; k *= 2531011u; }
    return k;
}

__host__ __device__ inline uint32_t gridHash(int type, const uint32_t* pos, int dims)
{
    const uint32_t prime[7] = {1958374283u, 2654435761u, 805459861u, 3674653429u, 2097192037u, 1434869437u, 2165219737u};
    switch (type) {
    case CV_HASH_PRIME: case CV_HASH_COHERENT_PRIME: case CV_HASH_REVERSED_PRIME: {   // lcgHash, :69-100
        uint32_t r = 0;
        for (int i = 0; i < dims; ++i) {
            uint32_t f = type == CV_HASH_REVERSED_PRIME ? prime[6 - i] : prime[i];
            if (type == CV_HASH_COHERENT_PRIME && i == 0) f = 1u;
            r ^= pos[i] * f;
        }
        return r; }
    case CV_HASH_RNG: {                                                // :117-131
        const int bits = 64 / dims;
        uint64_t step = 0;
        for (int i = 0; i < dims; ++i) step ^= (uint64_t)pos[i] << (i * bits);
        Pcg32 rng;
        rng.init(1337);
        rng.advance((int64_t)step);
        return rng.next(); }
    case CV_HASH_BASE_CONVERT: return baseConvertHash(pos, dims);
    }
    return 0;
}

__global__ __launch_bounds__(256) void gridHashKernel(int type, int dims, const uint8_t* pos, uint64_t stride, uint32_t* out, uint32_t batch)
{
    const uint32_t s = blockIdx.x * 256u + threadIdx.x;
    if (s >= batch) return;
    uint32_t p[7];
    for (int i = 0; i < dims; ++i) p[i] = ((const uint32_t*)(pos + (size_t)s * stride))[i];
    out[s] = gridHash(type, p, dims);
}

// ---- permutohedral lattice --------------------------------------------------------------------
struct PermutoArgs {
    CvPermutoDesc desc;
    const uint8_t* pos; uint64_t posStride;
    const uint8_t* table;
    uint8_t* out; uint64_t outStride;
    const uint8_t* dOut; uint64_t dOutStride;
    uint8_t* dPos; uint64_t dPosStride;
    float* dTable;
    uint32_t batch;
    float reach;      // latticeReach
};

template <typename T, int D>
__global__ __launch_bounds__(256) void permutoEncodeKernel(const PermutoArgs a)
{
    const uint32_t s = blockIdx.x * 256u + threadIdx.x;
    if (s >= a.batch) return;
    const int F = a.desc.featureDimensionPerEntry;
    float pos[D];
#pragma unroll
    for (int d = 0; d < D; ++d) pos[d] = (float)((const T*)(a.pos + (size_t)s * a.posStride))[d];
    T* out = (T*)(a.out + (size_t)s * a.outStride);
    const T* table = (const T*)a.table;
    for (uint32_t l = 0; l < a.desc.maxLevels; ++l) {
        const CvPermutoLevelInfo& lv = a.desc.levelInfo[l];
        T* o = out + lv.currentLevelIndex * F;
        for (int f = 0; f < F; ++f) o[f] = (T)0.f;
        if ((float)lv.currentLevelIndex >= a.desc.maxLevel + 1e-3f) continue;   // zero padding beyond maxLevel, :259-262
        LatticeSimplexAny<D> simplex;
        simplex.search(pos, latticeLevel<D>(lv));
        uint32_t idx[D + 1];
#pragma unroll
        for (int k = 0; k <= D; ++k) idx[k] = (lv.offsetOfFeatureTable + vertexSlot<false>(lv.featureTableSize, simplex.hash[k])) * (uint32_t)F;
        for (int f0 = 0; f0 < F; f0 += 4) {                            // four features of the entry at a time
            T acc[4] = {(T)0.f, (T)0.f, (T)0.f, (T)0.f};
#pragma unroll
            for (int k = 0; k <= D; ++k) {
                const T w = (T)simplex.bary[k];
#pragma unroll
                for (int f = 0; f < 4; ++f)
                    if (f0 + f < F) acc[f] = (T)(acc[f] + (T)(w * table[idx[k] + f0 + f]));    // in T, vertex by vertex (:312-316)
            }
#pragma unroll
            for (int f = 0; f < 4; ++f)
                if (f0 + f < F) o[f0 + f] = acc[f];
        }
    }
}

// The same encoding with one thread per (position, level), the level running fastest: a wave's 64 results are
// consecutive in memory (one thread per position writes F elements at the pitch of a whole row, which the memory
// system does not merge: 2.1 bytes written per byte of output), no thread loops over levels, and a feature table that
// fits is held in LDS, where a gather of 64 scattered entries costs a few cycles instead of one cache line per lane.
// The arithmetic per (position, level) is that of permutoEncodeKernel, bit for bit.
template <typename T, int D, int F, bool LDS_TABLE, bool PLAIN>
__global__ __launch_bounds__(1024) void permutoEncodePairsKernel(const PermutoArgs a, uint32_t tableElems, uint32_t levelShift)
{
    typedef typename PermutoEntry<T, F>::type Entry;
    extern __shared__ __align__(16) uint8_t ldsRaw[];
    static_assert(sizeof(LatticeLevel<D>) <= sizeof(CvPermutoLevelInfo), "the records' room in LDS is that of the description's");
    LatticeLevel<D>* levels = (LatticeLevel<D>*)ldsRaw;
    const T* ldsTable = (const T*)(ldsRaw + kMaxLevels * sizeof(CvPermutoLevelInfo));
    const uint32_t L = a.desc.maxLevels;
    {
        if (threadIdx.x < L) levels[threadIdx.x] = latticeLevel<D>(a.desc.levelInfo[threadIdx.x]);
        if constexpr (LDS_TABLE) {
            const Entry* t = (const Entry*)a.table;
            Entry* dst = (Entry*)(ldsRaw + kMaxLevels * sizeof(CvPermutoLevelInfo));
            for (uint32_t i = threadIdx.x; i < tableElems / (uint32_t)F; i += blockDim.x) dst[i] = t[i];
        }
    }
    __syncthreads();
    const T* table = LDS_TABLE ? ldsTable : (const T*)a.table;
    const uint64_t pairs = (uint64_t)a.batch * L;
    for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < pairs; p += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t s = levelShift < 32u ? (uint32_t)(p >> levelShift) : (uint32_t)(p / L);
        const uint32_t l = (uint32_t)(p - (uint64_t)s * L);
        const LatticeLevel<D>& lv = levels[l];
        float pos[D];
#pragma unroll
        for (int d = 0; d < D; ++d) pos[d] = (float)((const T*)(a.pos + (size_t)s * a.posStride))[d];
        Entry acc;
        if (!PLAIN || anyBeyondReach<D>(pos, a.reach)) acc = permutoEncodeEntry<T, D, F, PLAIN, LatticeSimplexAny<D>>(pos, lv, table, a.desc.maxLevel);
        else if constexpr (PLAIN) acc = permutoEncodeEntry<T, D, F, PLAIN, LatticeSimplex<D>>(pos, lv, table, a.desc.maxLevel);
        // (a streaming store: the encoded vectors are written once and read by the next kernel)
        __builtin_nontemporal_store(acc, (Entry*)((T*)(a.out + (size_t)s * a.outStride) + lv.index * F));
    }
}

// Where a position's contributions to the table gradient go: nowhere (position gradients only), straight to memory, or to
// a workgroup's copy of a part of the table in LDS.
struct NoTable {
    static constexpr bool kWanted = false;
    template <int N> __device__ __forceinline__ void addEntry(uint32_t, float, const float*) const {}
    __device__ __forceinline__ void add(uint32_t, int, float) const {}
};
struct TableInMemory {
    static constexpr bool kWanted = true;
    float* table;
    // w * g[0..N) to the entry whose first element is idx
    template <int N> __device__ __forceinline__ void addEntry(uint32_t idx, float w, const float* g) const
    {
#pragma unroll
        for (int f = 0; f < N; ++f) add(idx, f, w * g[f]);
    }
    __device__ __forceinline__ void add(uint32_t idx, int f, float v) const { atomicAdd(table + idx + f, v); }
};
// Elements [base, base + elems) of the table.  SLICED: what lies outside belongs to another workgroup.  The features of an
// entry are `entries` elements apart, so that one instruction's lanes, which add to the same feature of scattered entries,
// use all banks.
template <int FT, bool SLICED>
struct TableInLds {
    static constexpr bool kWanted = true;
    double* lds;
    uint32_t base, elems, entries, F;
    // Odd lanes begin with the last feature: on a coarse level, where a wave's positions share a few entries, half as many
    // lanes of an instruction meet on one address (25 entries in use: 57 -> 48 us for 2^18 positions on 8 such levels).
    template <int N> __device__ __forceinline__ void addEntry(uint32_t idx, float w, const float* g) const
    {
        const uint32_t e = idx - base;
        if (SLICED && e >= elems) return;
        const bool odd = N > 1 && (threadIdx.x & 1u);
        double* p = lds + e / (uint32_t)N + (odd ? (uint32_t)(N - 1) * entries : 0u);
        const int step = odd ? -(int)entries : (int)entries;
#pragma unroll
        for (int f = 0; f < N; ++f, p += step) unsafeAtomicAdd(p, (double)(w * (odd ? g[N - 1 - f] : g[f])));      // ds_add_f64
    }
    __device__ __forceinline__ void add(uint32_t idx, int f, float v) const
    {
        const uint32_t e = idx - base;
        if (!SLICED || e < elems) unsafeAtomicAdd(lds + (uint32_t)f * entries + e / F, (double)v);
    }
};

// Reverse mode of levels [first, end) for one position: hands bary[k] * dOut to `sink` and, with POS, writes the position
// gradient (of all levels: such calls take them all).
// FT: the features per entry when they are 1, 2 or 4 (the loops over them unrolled, the loads of a level issued together:
// with a run-time count every element was a load and a wait of its own), else 0.
// PLAIN, Simplex: as in permutoEncodeEntry.
template <int D, int FT, bool POS, bool PLAIN, typename Simplex, typename Sink>
__device__ __forceinline__ void permutoBackwardLevels(const PermutoArgs& a, const float* pos, uint32_t s, uint32_t first, uint32_t end, const Sink& sink)
{
    const int F = FT ? FT : a.desc.featureDimensionPerEntry;
    float dpos[D];
#pragma unroll
    for (int d = 0; d < D; ++d) dpos[d] = 0.f;
    const float* table = (const float*)a.table;
    const float* g = (const float*)(a.dOut + (size_t)s * a.dOutStride);
    for (uint32_t l = first; l < end; ++l) {
        const CvPermutoLevelInfo& lv = a.desc.levelInfo[l];
        if (!PLAIN && (float)lv.currentLevelIndex >= a.desc.maxLevel + 1e-3f) continue;
        Simplex simplex;
        simplex.search(pos, latticeLevel<D>(lv));
        float dbary[D + 1];
        uint32_t idx[D + 1];
#pragma unroll
        for (int k = 0; k <= D; ++k) {
            dbary[k] = 0.f;
            idx[k] = (lv.offsetOfFeatureTable + vertexSlot<PLAIN>(lv.featureTableSize, simplex.hash[k])) * (uint32_t)F;
        }
        const float* gl = g + lv.currentLevelIndex * F;
        if constexpr (FT > 0) {
            float gv[FT], tv[D + 1][FT];
#pragma unroll
            for (int f = 0; f < FT; ++f) gv[f] = gl[f];
            if constexpr (POS) {
#pragma unroll
                for (int k = 0; k <= D; ++k)
#pragma unroll
                    for (int f = 0; f < FT; ++f) tv[k][f] = table[idx[k] + f];
            }
#pragma unroll
            for (int k = 0; k <= D; ++k) {
                if constexpr (Sink::kWanted) sink.template addEntry<FT>(idx[k], simplex.bary[k], gv);    // readFeatureValueBwd, :222-238
#pragma unroll
                for (int f = 0; f < FT; ++f) {
                    if constexpr (POS) dbary[k] += tv[k][f] * gv[f];
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k <= D; ++k) {
                for (int f = 0; f < F; ++f) {
                    if constexpr (Sink::kWanted) sink.add(idx[k], f, simplex.bary[k] * gl[f]);    // readFeatureValueBwd, :222-238
                    if constexpr (POS) dbary[k] += table[idx[k] + f] * gl[f];
                }
            }
        }
        if constexpr (!POS) continue;
        float delev[D + 1];
        simplex.toElevated(dbary, delev);
        // elevate: e[dim+1] = sum - (dim+1) cf, sum += cf for dim = D-1..0, e[0] = sum
        float dsum = delev[0];
#pragma unroll
        for (int dim = 0; dim < D; ++dim) {
            const float dcf = dsum - (float)(dim + 1) * delev[dim + 1];
            dsum += delev[dim + 1];
            dpos[dim] += dcf * lv.scalesPerDim[dim];
        }
    }
    if constexpr (POS) {
#pragma unroll
        for (int d = 0; d < D; ++d) ((float*)(a.dPos + (size_t)s * a.dPosStride))[d] = dpos[d];
    }
}

template <int D, int FT, bool POS, bool PLAIN, typename Sink>
__device__ __forceinline__ void permutoBackwardOne(const PermutoArgs& a, uint32_t s, uint32_t first, uint32_t end, const Sink& sink)
{
    float pos[D];
#pragma unroll
    for (int d = 0; d < D; ++d) pos[d] = ((const float*)(a.pos + (size_t)s * a.posStride))[d];
    if constexpr (PLAIN) {
        if (!anyBeyondReach<D>(pos, a.reach)) {
            permutoBackwardLevels<D, FT, POS, true, LatticeSimplex<D>>(a, pos, s, first, end, sink);
            return;
        }
    }
    permutoBackwardLevels<D, FT, POS, PLAIN, LatticeSimplexAny<D>>(a, pos, s, first, end, sink);
}

// Position gradients alone (TABLE false), or everything with the table's share added in memory: a table of which one level
// alone is beyond what the LDS kernel below takes, or a handful of positions (launchBackwardSized).
template <int D, int FT, bool POS, bool TABLE, bool PLAIN>
__global__ __launch_bounds__(256) void permutoBackwardKernel(const PermutoArgs a)
{
    const uint32_t s = blockIdx.x * 256u + threadIdx.x;
    if (s >= a.batch) return;
    if constexpr (TABLE) permutoBackwardOne<D, FT, POS, PLAIN>(a, s, 0u, a.desc.maxLevels, TableInMemory{a.dTable});
    else permutoBackwardOne<D, FT, POS, PLAIN>(a, s, 0u, a.desc.maxLevels, NoTable{});
}

// The table gradient, by parts of the table small enough for LDS: part p covers elements [base, base + elems), which
// levels [first, end) add to.  Every position adds to a handful of entries per level; added in memory, where many positions
// meet on few addresses, 2^18 positions in 3 dimensions on 8 levels of 2^12 two-feature entries took 6.6 ms (2.5 G additions
// per second); here 36 us, of which a quarter is the start and the sums' way to memory.  (cutTable: cv_permuto_parts.h)
static_assert(sizeof(PermutoArgs) + sizeof(TableParts) <= 4096, "kernel arguments");

// A workgroup owns one part and a share of the positions: it sums into LDS and adds its sums to memory once, coalesced
// (180 G additions per second).  What bounds it: the LDS's additions and entries gathered from
// memory (with the position gradients beside it, 40 us, the waves of that case wait 48 % of their time for operands and 15 % for the LDS
// to take an instruction; the 351 vector instructions per position and level of both walks take 44 % of the port).  The sums are kept in double:
// at random addresses gfx950 serves a ds_add_f64 in 8.6 ns per wave and compute unit and a ds_add_f32 in 80 (16 waves), so the
// wider sum is also the cheaper one.  Lanes that meet on one address are served one after the other: 24 ns per LDS instruction
// in that case, 41 ns on the few entries of four coarse levels in two dimensions (2^22 positions: 256 us).
// POS: kPosInPass (one part that is the whole table), the position gradient in the same pass; kPosBeside (several parts), in
// passes of its own over all levels, whose units of 64 positions are dealt to the waves of all workgroups.  The two kinds of work
// wait for different things, additions in LDS and entries gathered from memory (64 lines each), so they go side by side: a
// workgroup's first waves take its units of positions and the others that much more of the table's (2^18 positions in 3
// dimensions, 8 levels of 2^12 two-feature entries: 40 us; 54.5 with the positions as a kernel of their own behind this one).  SLICED: some part is a slice of a level.
constexpr int kPosNone = 0, kPosInPass = 1, kPosBeside = 2;
// WAVES: on a SIMD; eight where two workgroups share a compute unit (64 registers a wave, two to thirteen of which spill in four
// dimensions or with four features and positions in the same pass), else four.
template <int D, int FT, int POS, bool SLICED, bool PLAIN, int WAVES>
__global__ __launch_bounds__(1024, WAVES) void permutoTableGradKernel(const PermutoArgs a, const TableParts parts)
{
    extern __shared__ double ldsTable[];
    // workgroup w: part w / groups, so that the workgroups of all parts that read the same positions (w % groups) sit on one
    // die (w % 8) where groups is a multiple of 8, and find them in its L2
    const uint32_t p = blockIdx.x / parts.groups, w = blockIdx.x - p * parts.groups;
    const TablePart part = parts.part[p];
    const uint32_t F = FT ? (uint32_t)FT : (uint32_t)a.desc.featureDimensionPerEntry, entries = part.elems / F;
    for (uint32_t i = threadIdx.x; i < part.elems; i += 1024u) ldsTable[i] = 0.0;
    __syncthreads();
    const TableInLds<FT, SLICED> sink{ldsTable, part.base, part.elems, entries, F};
    if constexpr (POS != kPosBeside) {
        // units of 64 positions, dealt to the part's workgroups in turn
        for (uint64_t s = ((uint64_t)(threadIdx.x >> 6) * parts.groups + w) * 64u + (threadIdx.x & 63u); s < a.batch; s += (uint64_t)parts.groups * 1024u)
            permutoBackwardOne<D, FT, POS == kPosInPass, PLAIN>(a, (uint32_t)s, part.first, part.end, sink);
    } else {
        const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63u;
        const uint32_t units = (a.batch - 1u) / 64u + 1u;
        for (uint64_t u = (uint64_t)wave * gridDim.x + blockIdx.x; u < units; u += 16ull * gridDim.x) {
            const uint64_t s = u * 64u + lane;
            if (s < a.batch) permutoBackwardOne<D, FT, true, PLAIN>(a, (uint32_t)s, 0u, a.desc.maxLevels, NoTable{});
        }
        // of this workgroup's units of positions (one by one to the waves) the first `more` waves have one more than the others,
        // which for that take `worth` units of the table ahead of everyone's turns
        const uint32_t own = blockIdx.x < units ? (units - 1u - blockIdx.x) / gridDim.x + 1u : 0u;
        const uint32_t more = own % 16u, worth = more ? a.desc.maxLevels / (part.end - part.first) : 0u;
        const uint32_t ahead = (16u - more) * worth;
        const uint32_t turns = wave >= more ? worth : 0u;
        for (uint32_t i = 0;; ++i) {
            const uint64_t t = i < turns ? (wave - more) + (uint64_t)i * (16u - more) : ahead + wave + 16ull * (i - turns);
            const uint64_t u = t * parts.groups + w, s = u * 64u + lane;
            if (u >= units) break;           // (t grows with i)
            if (s < a.batch) permutoBackwardOne<D, FT, false, PLAIN>(a, (uint32_t)s, part.first, part.end, sink);
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < part.elems; i += 1024u) {
        const uint32_t e = i / F, f = i - e * F;
        const float v = (float)ldsTable[f * entries + e];
        if (v != 0.f) atomicAdd(a.dTable + part.base + i, v);
    }
}

// the table as the levels lay it out: offsets and sizes in entries, F elements per entry
uint64_t tableElements(const CvPermutoDesc& d)
{
    uint64_t n = 0;
    for (uint32_t l = 0; l < d.maxLevels; ++l) {
        const uint64_t e = ((uint64_t)d.levelInfo[l].offsetOfFeatureTable + d.levelInfo[l].featureTableSize) * (uint64_t)d.featureDimensionPerEntry;
        n = e > n ? e : n;
    }
    return n;
}

constexpr size_t kPairsLevelBytes = kMaxLevels * sizeof(CvPermutoLevelInfo);
constexpr size_t kPairsTableBytes = 144 * 1024;      // with the level records: within the 160 KB of a compute unit

template <typename T, int D, int F>
hipError_t launchEncodePairs(hipStream_t stream, const PermutoArgs& a)
{
    const uint64_t tableElems = tableElements(a.desc);
    const bool inLds = tableElems * sizeof(T) <= kPairsTableBytes;
    const size_t lds = kPairsLevelBytes + (inLds ? (size_t)tableElems * sizeof(T) : 0);
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    const uint64_t pairs = (uint64_t)a.batch * a.desc.maxLevels, want = (pairs + 1023u) / 1024u;
    const uint64_t cap = (uint64_t)cus * (lds <= 80 * 1024 ? 2u : 1u);
    const dim3 grid((uint32_t)(want < cap ? want : cap)), block(1024);
    const uint32_t L = a.desc.maxLevels;
    const uint32_t shift = (L & (L - 1u)) == 0u ? (uint32_t)__builtin_ctz(L) : 0xffffffffu;
    auto launch = [&](auto plainConst) -> hipError_t {
        constexpr bool PLAIN = decltype(plainConst)::value;
        if (inLds) {
            const hipError_t e = allowDynamicLds<permutoEncodePairsKernel<T, D, F, true, PLAIN>>((int)(kPairsLevelBytes + kPairsTableBytes));
            if (e != hipSuccess) return e;
            hipLaunchKernelGGL((permutoEncodePairsKernel<T, D, F, true, PLAIN>), grid, block, lds, stream, a, (uint32_t)tableElems, shift);
        } else {
            hipLaunchKernelGGL((permutoEncodePairsKernel<T, D, F, false, PLAIN>), grid, block, lds, stream, a, (uint32_t)tableElems, shift);
        }
        return hipGetLastError();
    };
    return permutoPlainLevels(a.desc) ? launch(std::true_type()) : launch(std::false_type());
}

// the kernel above takes entries of 4, 8 or 16 bytes at addresses that are multiples of their size
template <typename T>
bool pairsEligible(const PermutoArgs& a)
{
    const size_t eb = (size_t)a.desc.featureDimensionPerEntry * sizeof(T);
    const int F = a.desc.featureDimensionPerEntry;
    if (a.desc.dimensions > 4 || (F != 1 && F != 2 && F != 4 && F != 8) || eb > 16) return false;
    return (uintptr_t)a.table % eb == 0 && (uintptr_t)a.out % eb == 0 && a.outStride % eb == 0 && tableElements(a.desc) <= 0xffffffffull;
}

template <typename T>
hipError_t launchEncode(hipStream_t stream, const PermutoArgs& a)
{
    if (pairsEligible<T>(a)) {
        noteKernel(false, "permutoEncodePairsKernel<%s,D=%d,F=%d>", sizeof(T) == 4 ? "f32" : "f16", a.desc.dimensions, a.desc.featureDimensionPerEntry);
        switch (a.desc.dimensions * 16 + a.desc.featureDimensionPerEntry) {
#define CV_DF(N, G) case N * 16 + G: if constexpr (G * sizeof(T) <= 16) return launchEncodePairs<T, N, G>(stream, a); break;
        CV_DF(1, 1) CV_DF(1, 2) CV_DF(1, 4) CV_DF(1, 8) CV_DF(2, 1) CV_DF(2, 2) CV_DF(2, 4) CV_DF(2, 8)
        CV_DF(3, 1) CV_DF(3, 2) CV_DF(3, 4) CV_DF(3, 8) CV_DF(4, 1) CV_DF(4, 2) CV_DF(4, 4) CV_DF(4, 8)
#undef CV_DF
        }
    }
    noteKernel(false, "permutoEncodeKernel<%s,D=%d>", sizeof(T) == 4 ? "f32" : "f16", a.desc.dimensions);
    const dim3 grid((a.batch + 255) / 256), block(256);
    switch (a.desc.dimensions) {
#define CV_D(N) case N: hipLaunchKernelGGL((permutoEncodeKernel<T, N>), grid, block, 0, stream, a); break;
    CV_D(1) CV_D(2) CV_D(3) CV_D(4) CV_D(5) CV_D(6) CV_D(7) CV_D(8)
#undef CV_D
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int D, int FT, int POS, bool SLICED, bool PLAIN, int WAVES>
hipError_t launchTableGradWaves(hipStream_t stream, const PermutoArgs& a, const TableParts& t)
{
    const hipError_t e = allowDynamicLds<permutoTableGradKernel<D, FT, POS, SLICED, PLAIN, WAVES>>((int)(kPartMost * 8));
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((permutoTableGradKernel<D, FT, POS, SLICED, PLAIN, WAVES>), dim3(t.count * t.groups), dim3(1024), (size_t)largestPart(t) * 8, stream, a, t);
    return hipGetLastError();
}
template <int D, int FT, int POS, bool SLICED, bool PLAIN>
hipError_t launchTableGrad(hipStream_t stream, const PermutoArgs& a, const TableParts& t, int cus)
{
    constexpr bool kSmall = D <= 4 && FT > 0;
    // (one part, table and positions in a pass: 64 registers are too few for some, so a table or a batch that puts one workgroup on a
    // compute unit has twice as many; 4 dimensions, one level of 2^12 four-feature entries, 2^18 positions: 22.4 -> 20.9 us)
    if constexpr (kSmall && POS == kPosInPass) {
        if (largestPart(t) > kPartHalf || t.count * t.groups <= (uint32_t)cus) return launchTableGradWaves<D, FT, POS, SLICED, PLAIN, 4>(stream, a, t);
    }
    return launchTableGradWaves<D, FT, POS, SLICED, PLAIN, kSmall ? 8 : 4>(stream, a, t);
}

template <int D, int FT, bool PLAIN>
hipError_t launchBackwardLevels(hipStream_t stream, const PermutoArgs& a)
{
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    const dim3 grid((a.batch - 1u) / 256u + 1u), block(256);
    const uint64_t features = (uint64_t)a.desc.featureDimensionPerEntry * a.desc.maxLevels;
    // Where position gradients are written on top of what is read (rows on rows), other workgroups of one launch would still read it.
    const Rows dPos{(uint64_t)(uintptr_t)a.dPos, a.dPosStride, D * 4ull}, pos{(uint64_t)(uintptr_t)a.pos, a.posStride, D * 4ull},
        dOut{(uint64_t)(uintptr_t)a.dOut, a.dOutStride, features * 4ull};
    const bool apart = a.dPos && !rowsMeet(dPos, pos, a.batch) && !rowsMeet(dPos, dOut, a.batch);
    TableParts t;
    const bool cut = a.dTable && planTable(a.desc, a.batch, (uint32_t)cus, FT > 0 && (apart || !a.dPos), t);
    if (cut && t.count == 1 && a.dPos) {
        noteKernel(false, "permutoTableGradKernel<D=%d,positions>", D);
        return launchTableGrad<D, FT, kPosInPass, false, PLAIN>(stream, a, t, cus);
    }
    // A handful of positions whose few additions hardly meet is done sooner by the one kernel that adds in memory: 4.1 to 4.7 us where the
    // table in slices, which takes two launches, has 7.9 (4 levels of 2^15 entries, 1 to 64 positions).  Its time grows with the additions and
    // reaches the two launches' at 1300 to 2000 of them.  Against one launch it is the sooner one up to 580 to 860 additions (3 levels of 2^10
    // four-feature entries, 16 / 24 / 32 positions 4.7, 6.8, 8.3 against 5.8, 5.7, 5.7; 2 of 2^12 two-feature ones, 24 / 32 / 48 4.2, 5.1, 6.7 against 5.2),
    // or beyond 1440 where they spread over more entries (4 dimensions, 6 levels of 2^12, 48 positions 7.4 against 8.4; 4 levels of 2^12
    // four-feature entries, 16 positions 6.2 against 7.8): no line by their number serves both, so there is one for all.  Where a position has more than 16 features it
    // is the slower one from the first position (16 levels of 4 features: 34.8 against 14.5 us).
    const bool few = FT > 0 && a.batch <= 64u && features <= 16u && a.batch * (uint64_t)(D + 1) * features <= 1440u;
    if (cut && !(a.dPos && few)) {
        if (apart && positionsBeside(t, a.batch, (uint32_t)cus)) {      // (one launch)
            noteKernel(false, "permutoTableGradKernel<D=%d,%u parts,positions beside>", D, t.count);
            return t.sliced ? launchTableGrad<D, FT, kPosBeside, true, PLAIN>(stream, a, t, cus) : launchTableGrad<D, FT, kPosBeside, false, PLAIN>(stream, a, t, cus);
        }
        noteKernel(false, "permutoTableGradKernel<D=%d,%u parts>", D, t.count);
        const hipError_t e = t.sliced ? launchTableGrad<D, FT, kPosNone, true, PLAIN>(stream, a, t, cus) : launchTableGrad<D, FT, kPosNone, false, PLAIN>(stream, a, t, cus);
        if (e != hipSuccess || !a.dPos) return e;
        noteKernel(true, "permutoBackwardKernel<D=%d,positions>", D);
        hipLaunchKernelGGL((permutoBackwardKernel<D, FT, true, false, PLAIN>), grid, block, 0, stream, a);
        return hipGetLastError();
    }
    noteKernel(false, "permutoBackwardKernel<D=%d%s%s>", D, a.dPos ? ",positions" : "", a.dTable ? ",table" : "");
    if (a.dPos && a.dTable) hipLaunchKernelGGL((permutoBackwardKernel<D, FT, true, true, PLAIN>), grid, block, 0, stream, a);
    else if (a.dPos) hipLaunchKernelGGL((permutoBackwardKernel<D, FT, true, false, PLAIN>), grid, block, 0, stream, a);
    else if (a.dTable) hipLaunchKernelGGL((permutoBackwardKernel<D, FT, false, true, PLAIN>), grid, block, 0, stream, a);
    return hipGetLastError();
}

// (kernels of their own for plain levels where vectors of few dimensions and entries of 1, 2 or 4 features make them worth
// their code)
template <int D, int FT>
hipError_t launchBackwardSized(hipStream_t stream, const PermutoArgs& a)
{
    if constexpr (D <= 4 && FT > 0) {
        if (permutoPlainLevels(a.desc)) return launchBackwardLevels<D, FT, true>(stream, a);
    }
    return launchBackwardLevels<D, FT, false>(stream, a);
}

hipError_t launchBackward(hipStream_t stream, const PermutoArgs& a)
{
    const int fe = a.desc.featureDimensionPerEntry, ft = (fe == 1 || fe == 2 || fe == 4) ? fe : 0;
    switch (a.desc.dimensions * 8 + ft) {
#define CV_DF(N, G) case N * 8 + G: return launchBackwardSized<N, G>(stream, a);
#define CV_D(N) CV_DF(N, 0) CV_DF(N, 1) CV_DF(N, 2) CV_DF(N, 4)
    CV_D(1) CV_D(2) CV_D(3) CV_D(4) CV_D(5) CV_D(6) CV_D(7) CV_D(8)
#undef CV_D
#undef CV_DF
    }
    return hipErrorInvalidValue;
}

} // namespace

CvResult checkPermutoDesc(const char* who, const CvPermutoDesc* d)
{
    if (!d) return failWith(CV_E_INVALID_ARG, "%s: desc is null", who);
    if (d->dimensions < 1 || d->dimensions > kMaxDims) return failWith(CV_E_INVALID_ARG, "%s: dimensions=%d (1..%d)", who, d->dimensions, kMaxDims);
    if (d->featureDimensionPerEntry < 1 || d->featureDimensionPerEntry > 64)
        return failWith(CV_E_INVALID_ARG, "%s: featureDimensionPerEntry=%d (1..64)", who, d->featureDimensionPerEntry);
    if (d->maxLevels < 1 || d->maxLevels > (uint32_t)kMaxLevels) return failWith(CV_E_INVALID_ARG, "%s: maxLevels=%u (1..%d)", who, d->maxLevels, kMaxLevels);
    if (d->elementType != CV_FLOAT32 && d->elementType != CV_FLOAT16)
        return failWith(CV_E_NOT_AVAILABLE, "%s: elementType %d (supported: FLOAT32, FLOAT16)", who, d->elementType);
    for (uint32_t l = 0; l < d->maxLevels; ++l)
        if (d->levelInfo[l].featureTableSize == 0 || d->levelInfo[l].currentLevelIndex >= d->maxLevels)
            return failWith(CV_E_INVALID_ARG, "%s: level %u: empty feature table or level index %u out of range", who, l, d->levelInfo[l].currentLevelIndex);
    return CV_OK;
}

} // namespace cv

extern "C" {

CV_API CvResult cvGridHash(void* stream, int32_t hashType, int32_t dimensions, const void* positions, size_t positionStride,
                           uint32_t* out, uint32_t batch)
{
    using namespace cv;
    if (hashType < CV_HASH_PRIME || hashType > CV_HASH_BASE_CONVERT) return failWith(CV_E_INVALID_ARG, "cvGridHash: unknown hash type %d", hashType);
    if (dimensions < 1 || dimensions > 7) return failWith(CV_E_INVALID_ARG, "cvGridHash: dimensions=%d (1..7, the prime table of the reference)", dimensions);
    if (batch == 0) return CV_OK;
    if (!positions || !out || (uintptr_t)positions % 4 || positionStride % 4 || (uintptr_t)out % 4 ||
        (batch > 1 && positionStride < (size_t)dimensions * 4))
        return failWith(CV_E_INVALID_ARG, "cvGridHash: null or misaligned argument");
    noteKernel(false, "gridHashKernel");
    hipLaunchKernelGGL(gridHashKernel, dim3((batch + 255) / 256), dim3(256), 0, (hipStream_t)stream, hashType, dimensions,
                       (const uint8_t*)positions, (uint64_t)positionStride, out, batch);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return failWith(CV_E_INTERNAL_FAIL, "cvGridHash launch: %s", hipGetErrorString(e));
    return CV_OK;
}

CV_API CvResult cvPermutoPrepareLevels(CvPermutoDesc* d, float baseScale, float log2PerLevelScale, float maxLevelRatio, uint32_t seed)
{
    using namespace cv;
    if (!d) return failWith(CV_E_INVALID_ARG, "cvPermutoPrepareLevels: desc is null");
    if (d->dimensions < 1 || d->dimensions > kMaxDims || d->maxLevels < 1 || d->maxLevels > (uint32_t)kMaxLevels || d->log2HashmapSize > 30)
        return failWith(CV_E_INVALID_ARG, "cvPermutoPrepareLevels: dimensions=%d maxLevels=%u log2HashmapSize=%u", d->dimensions, d->maxLevels, d->log2HashmapSize);
    const uint32_t size = 1u << d->log2HashmapSize;
    d->maxLevel = maxLevelRatio * (float)d->maxLevels;
    for (uint32_t level = 0; level < d->maxLevels; ++level) {          // prepareLevelInfo, permuto-encoder.slang:339-368
        CvPermutoLevelInfo& lv = d->levelInfo[level];
        memset(&lv, 0, sizeof(lv));
        lv.currentLevelIndex = level;
        lv.featureTableSize = size;
        lv.offsetOfFeatureTable = level * size;
        lv.scale = baseScale * exp2f((float)level * log2PerLevelScale);
        Pcg32 rng;
        rng.init(seed);
        rng.advance((int64_t)(level * (uint32_t)d->dimensions));
        for (int dim = 0; dim < d->dimensions; ++dim) {
            lv.scalesPerDim[dim] = lv.scale * (1.0f / sqrtf((float)((dim + 1) * (dim + 2))));
            const float r = (float)rng.next() * (1.0f / 4294967296.0f);
            lv.shiftsPerDim[dim] = r * 10.0f - 5.0f;
        }
    }
    return CV_OK;
}

CV_API CvResult cvPermutoEncode(void* stream, const CvPermutoDesc* desc, const void* positions, size_t positionStride,
                                const void* featureTable, void* out, size_t outStride, uint32_t batch)
{
    using namespace cv;
    CvResult rc = checkPermutoDesc("cvPermutoEncode", desc);
    if (CV_FAILED(rc)) return rc;
    if (batch == 0) return CV_OK;
    const uint32_t esz = desc->elementType == CV_FLOAT32 ? 4u : 2u;
    const size_t nOut = (size_t)desc->maxLevels * desc->featureDimensionPerEntry;
    if (!positions || !featureTable || !out || (uintptr_t)positions % esz || positionStride % esz || (uintptr_t)featureTable % esz ||
        (uintptr_t)out % esz || outStride % esz ||
        (batch > 1 && (positionStride < (size_t)desc->dimensions * esz || outStride < nOut * esz)))
        return failWith(CV_E_INVALID_ARG, "cvPermutoEncode: null, misaligned or overlapping-row argument");
    PermutoArgs a;
    memset(&a, 0, sizeof(a));
    a.desc = *desc;
    a.pos = (const uint8_t*)positions; a.posStride = positionStride; a.table = (const uint8_t*)featureTable;
    a.out = (uint8_t*)out; a.outStride = outStride; a.batch = batch; a.reach = latticeReach(*desc);
    const hipError_t e = esz == 4 ? launchEncode<float>((hipStream_t)stream, a) : launchEncode<half_t>((hipStream_t)stream, a);
    if (e != hipSuccess) return failWith(CV_E_INTERNAL_FAIL, "cvPermutoEncode launch: %s", hipGetErrorString(e));
    return CV_OK;
}

CV_API CvResult cvPermutoEncodeBackward(void* stream, const CvPermutoDesc* desc, const void* positions, size_t positionStride,
                                        const void* featureTable, const void* dOut, size_t dOutStride,
                                        void* dPositions, size_t dPositionStride, void* dFeatureTable, uint32_t batch)
{
    using namespace cv;
    CvResult rc = checkPermutoDesc("cvPermutoEncodeBackward", desc);
    if (CV_FAILED(rc)) return rc;
    if (desc->elementType != CV_FLOAT32)
        return failWith(CV_E_NOT_AVAILABLE, "cvPermutoEncodeBackward: FLOAT32 data only (the table gradient is accumulated with fp32 atomic adds)");
    if (batch == 0) return CV_OK;
    const size_t nOut = (size_t)desc->maxLevels * desc->featureDimensionPerEntry;
    if (!positions || !featureTable || !dOut || (uintptr_t)positions % 4 || positionStride % 4 || (uintptr_t)featureTable % 4 ||
        (uintptr_t)dOut % 4 || dOutStride % 4 || (uintptr_t)dPositions % 4 || dPositionStride % 4 || (uintptr_t)dFeatureTable % 4 ||
        (batch > 1 && (positionStride < (size_t)desc->dimensions * 4 || dOutStride < nOut * 4 ||
                       (dPositions && dPositionStride < (size_t)desc->dimensions * 4))))
        return failWith(CV_E_INVALID_ARG, "cvPermutoEncodeBackward: null, misaligned or overlapping-row argument");
    PermutoArgs a;
    memset(&a, 0, sizeof(a));
    a.desc = *desc;
    a.pos = (const uint8_t*)positions; a.posStride = positionStride; a.table = (const uint8_t*)featureTable;
    a.dOut = (const uint8_t*)dOut; a.dOutStride = dOutStride;
    a.dPos = (uint8_t*)dPositions; a.dPosStride = dPositionStride; a.dTable = (float*)dFeatureTable; a.batch = batch; a.reach = latticeReach(*desc);
    const hipError_t e = launchBackward((hipStream_t)stream, a);
    if (e != hipSuccess) return failWith(CV_E_INTERNAL_FAIL, "cvPermutoEncodeBackward launch: %s", hipGetErrorString(e));
    return CV_OK;
}

} // extern "C"
