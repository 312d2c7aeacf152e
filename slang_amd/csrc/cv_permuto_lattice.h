// cv_permuto_lattice.h -- the simplex of the permutohedral lattice that encloses a position: barycentric weights, vertex
// hashes, and the way back from gradients of the weights to gradients of the position.  Plain arithmetic, compiled for the
// GPU by the encoder kernels and for the host by the test that compares it with the steps as the reference writes them.
//
// What it restates: the per-level steps of PermutoEncoder::encode (source/standard-modules/neural/permuto-encoder.slang:240-337):
// elevate the position, find the closest remainder-0 lattice point and the ranks (:74-152), the barycentric weights
// (:166-179) and the keys of the D+1 vertices (:296-309).  Line numbers below refer to that file.
#pragma once
#include <cmath>
#include <cstdint>

#include "coopvec.h"

#if defined(__HIP__) || defined(__HIPCC__)
#define CV_LATTICE_FN __host__ __device__ __forceinline__
#else
#define CV_LATTICE_FN inline
#endif

namespace cv {

// The multipliers of baseConvertHash (sum key[d] * c^(D-d) modulo 2^32) and what they give per vertex.
template <int D>
struct LatticeHash {
    uint32_t mult[D + 1] = {}, all = 0;      // (the last dimension's key is not hashed: multiplier 0)
    constexpr LatticeHash()
    {
        uint32_t p = 2531011u;
        for (int d = D - 1; d >= 0; --d) { mult[d] = p; all += p; p *= 2531011u; }
    }
};

// One level's record as the kernels keep it (in LDS, or made from the description on the way): `unit` is the scale over D+1, which
// is exact where D+1 is a power of two and used only there.
template <int D>
struct LatticeLevel {
    float shift[D], scale[D], unit[D];
    uint32_t size, offset;                   // of the feature table, in entries
    uint32_t index;                          // currentLevelIndex
};
template <int D>
CV_LATTICE_FN LatticeLevel<D> latticeLevel(const CvPermutoLevelInfo& lv)
{
    LatticeLevel<D> r;
#pragma unroll
    for (int d = 0; d < D; ++d) {
        r.shift[d] = lv.shiftsPerDim[d];
        r.scale[d] = lv.scalesPerDim[d];
        r.unit[d] = lv.scalesPerDim[d] * (1.0f / (float)(D + 1));
    }
    r.size = lv.featureTableSize;
    r.offset = lv.offsetOfFeatureTable;
    r.index = lv.currentLevelIndex;
    return r;
}

// elevated coordinates (:74-84); scales and result may both be in units of D+1
template <int D>
CV_LATTICE_FN void elevate(const float* pos, const float* shift, const float* scale, float (&elevated)[D + 1])
{
    float sum = 0.0f;
#pragma unroll
    for (int dim = D - 1; dim >= 0; --dim) {
        const float cf = (pos[dim] + shift[dim]) * scale[dim];
        elevated[dim + 1] = dim == D - 1 ? (float)(dim + 1) * -cf : sum - (float)(dim + 1) * cf;
        sum = dim == D - 1 ? cf : sum + cf;
    }
    elevated[0] = sum;
}

// The steps as the reference has them, ranks counted and arrays in the order of ranks by selects: any position whatever.
template <int D>
struct LatticeSimplexAny {
    static constexpr int N = D + 1;
    float bary[N];                           // weight of the remainder-k vertex
    uint32_t hash[N];                        // of its key
    int rank[N];

    CV_LATTICE_FN void search(const float* pos, const LatticeLevel<D>& lv)
    {
        float elevated[N];
        elevate<D>(pos, lv.shift, lv.scale, elevated);
        int rem0[N], isum = 0;
#pragma unroll
        for (int dim = 0; dim < N; ++dim) {
            rank[dim] = 0;
            const float v = elevated[dim] * (1.0f / (float)N);
            const float up = __builtin_ceilf(v) * (float)N, down = __builtin_floorf(v) * (float)N;
            rem0[dim] = (up - elevated[dim] < elevated[dim] - down) ? (int)up : (int)down;
            isum += rem0[dim];
        }
        isum /= N;
#pragma unroll
        for (int dim = 0; dim < D; ++dim) {
            const float di = elevated[dim] - (float)rem0[dim];
#pragma unroll
            for (int other = dim + 1; other < N; ++other) {
                if (di < elevated[other] - (float)rem0[other]) rank[dim]++;
                else rank[other]++;
            }
        }
        float delta[N];
#pragma unroll
        for (int dim = 0; dim < N; ++dim) {
            rank[dim] += isum;
            const int wrap = rank[dim] < 0 ? N : (rank[dim] > D ? -N : 0);     // :146-156, as selects
            rank[dim] += wrap;
            rem0[dim] += wrap;
            delta[dim] = (elevated[dim] - (float)rem0[dim]) * (1.0f / (float)N);
        }
        // barycentric[D - rank] += delta, barycentric[D + 1 - rank] -= delta (:166-179)
        float sorted[N];
#pragma unroll
        for (int r = 0; r < N; ++r) {
            float v = delta[D];
#pragma unroll
            for (int dim = D - 1; dim >= 0; --dim) { const float own = delta[dim]; v = rank[dim] == r ? own : v; }
            sorted[r] = v;
        }
#pragma unroll
        for (int k = 1; k < N; ++k) bary[k] = (0.0f + sorted[D - k]) - sorted[D + 1 - k];
        bary[0] = (0.0f + sorted[D]) + (1.0f + (0.0f - sorted[0]));
        // the key of vertex k is rem0 + k, less N in the dimensions ranked above D - k (:296-303)
        constexpr LatticeHash<D> h;
        uint32_t key = 0u;
#pragma unroll
        for (int dim = 0; dim < D; ++dim) key += (uint32_t)rem0[dim] * h.mult[dim];
        hash[0] = key;
#pragma unroll
        for (int k = 1; k < N; ++k) {
            uint32_t less = 0u;
#pragma unroll
            for (int dim = 0; dim < D; ++dim) less = rank[dim] == N - k ? (uint32_t)N * h.mult[dim] : less;
            key += h.all - less;
            hash[k] = key;
        }
    }

    // gradients of the elevated coordinates from those of the weights
    CV_LATTICE_FN void toElevated(const float (&dbary)[N], float (&delev)[N]) const
    {
#pragma unroll
        for (int dim = 0; dim < N; ++dim) {
            float plus = 0.f, minus = 0.f;
#pragma unroll
            for (int i = 0; i <= N; ++i) {
                const float own = dbary[i % N];
                plus = i == D - rank[dim] ? own : plus;
                minus = i == N - rank[dim] ? own : minus;
            }
            delev[dim] = (plus - minus) * (1.0f / (float)N);
        }
    }
};

// The greatest |position| at which no level's elevated values exceed 2^22, the range of LatticeSimplex below; negative: none.
inline float latticeReach(const CvPermutoDesc& desc)
{
    float reach = 3.0e38f;
    for (uint32_t l = 0; l < desc.maxLevels; ++l) {
        float sum = 0.f, shift = 0.f;
        for (int d = 0; d < desc.dimensions; ++d) {
            const float scale = std::fabs(desc.levelInfo[l].scalesPerDim[d]), move = std::fabs(desc.levelInfo[l].shiftsPerDim[d]);
            if (!(scale < 1e30f) || !(move < 1e30f)) return -1.0f;
            sum += (float)(d + 2) * scale;                                   // |elevated| <= sum * (|position| + |shift|)
            shift = std::fmax(shift, move);
        }
        reach = std::fmin(reach, 4194304.0f / std::fmax(sum, 1e-30f) - shift);
    }
    return reach;
}

// The same bits with fewer instructions, for elevated values up to 2^22 (latticeReach).  What bounds the kernels that use it is
// vector-ALU issue, so the count is what matters: 3 dimensions, 225 instructions per position and level with the steps above,
// about 130 here (encoder of 8 levels and decoder 16-64-64-3 over 2^22 positions: 223 -> 169 us).
//
//   - d[dim] = elevated - rem0 is exact (the nearest multiple of N = D+1, so at most a factor of two away), hence
//     elevated - (rem0 +- N), the same after the wrap of :146-156, rounds to what d -+ N rounds to.  Where N is a power of two all
//     of this is computed in units of N, which scales every value exactly (elevated values below 2^-147 count as zero).
//   - The ranks are the stable descending order of d, then shifted by the sum s of the rounded quotients modulo N.  Here the
//     values themselves are put in order by exchanges that keep equal values in the order of their dimensions, each carrying the dimension's part of the hash; then turned by s.
//     Order k = 0..D below is ascending, rank D - k.
//   - The key of the remainder-(k+1) vertex is that of the remainder-k one plus 1, less N in the dimension of the next
//     lowest rank; the hash is linear, so it steps by a constant of that dimension.  N steps return to the start, so the
//     vertices before and after the turn are the same ring: V'[k] = V[(k + s) mod N] - s * (sum of the multipliers).
//
//   - Hashes count modulo 2^24, which the full-rate 24-bit multiplies give: for tables of 2^n entries, n <= 24.
template <int D>
struct LatticeSimplex {
    static_assert(D <= 4, "more dimensions are not worth their code");
    static constexpr int N = D + 1;
    static constexpr bool kPow2 = (N & (N - 1)) == 0;
    static constexpr int kTurnBits = N > 4 ? 3 : N > 2 ? 2 : 1;      // of a number below N

    // The x-th exchange is of positions exchangeAt(x) and exchangeAt(x) + apart(x).  Neighbours: in turn all even and all odd
    // ones, N - 1 exchanges for both.  Four values take five exchanges instead of six, (0,1) (2,3) (0,2) (1,3) (1,2): the first
    // four leave equal values in order, and behind them the last one exchanges equal values too, unless the two before it
    // did nothing (then positions 1 and 2 still hold a value of the first and a value of the second pair).
    static constexpr int kExchanges = N == 4 ? 5 : N * (N - 1) / 2;
    static constexpr int exchangeAt(int x) { return N == 4 ? (x == 1 ? 2 : x >= 3 ? 1 : 0) : x % D < N / 2 ? 2 * (x % D) : 2 * (x % D - N / 2) + 1; }
    static constexpr int apart(int x) { return N == 4 && (x == 2 || x == 3) ? 2 : 1; }

    // A condition in scalar registers, where combining two of them takes no vector instruction (of bools the compiler would go
    // back to the numbers they were tests of).
#if defined(__HIP_DEVICE_COMPILE__)
    typedef uint64_t Lanes;
    static CV_LATTICE_FN Lanes lanesOf(bool c) { Lanes m = __builtin_amdgcn_ballot_w64(c); asm("" : "+s"(m)); return m; }
    static CV_LATTICE_FN bool in(Lanes m) { return __builtin_amdgcn_inverse_ballot_w64(m); }
#else
    typedef bool Lanes;
    static CV_LATTICE_FN Lanes lanesOf(bool c) { return c; }
    static CV_LATTICE_FN bool in(Lanes m) { return m; }
#endif

    float bary[N];                           // weight of the remainder-k vertex
    uint32_t hash[N];                        // of its key, modulo 2^24 (the upper bits are any)
    Lanes turn[kTurnBits];                   // the bits of s modulo N
    bool exchanged[kExchanges];              // the exchanges that put the dimensions in order

    // x[k] = x[(k + by) mod N], by < N, as a few selects per bit of `by`.  (Both values are read before the choice, here and
    // below: a choice between elements of an array would become an element at a chosen index.)
    template <typename V>
    static CV_LATTICE_FN void turnBy(V (&x)[N], const Lanes (&by)[kTurnBits])
    {
#pragma unroll
        for (int i = 0; i < kTurnBits; ++i) {
            const int b = 1 << i;
            const bool on = in(by[i]);
            V y[N];
#pragma unroll
            for (int k = 0; k < N; ++k) { const V from = x[(k + b) % N], own = x[k]; y[k] = on ? from : own; }
#pragma unroll
            for (int k = 0; k < N; ++k) x[k] = y[k];
        }
    }
    template <typename V>
    static CV_LATTICE_FN void turnBack(V (&x)[N], const Lanes (&by)[kTurnBits])
    {
#pragma unroll
        for (int i = 0; i < kTurnBits; ++i) {
            const int b = 1 << i;
            const bool on = in(by[i]);
            V y[N];
#pragma unroll
            for (int k = 0; k < N; ++k) { const V from = x[(k + N - b) % N], own = x[k]; y[k] = on ? from : own; }
#pragma unroll
            for (int k = 0; k < N; ++k) x[k] = y[k];
        }
    }
    CV_LATTICE_FN void search(const float* pos, const LatticeLevel<D>& lv)
    {
        constexpr LatticeHash<D> h;
        float elevated[N];
        elevate<D>(pos, lv.shift, kPow2 ? lv.unit : lv.scale, elevated);

        // d[k] and hash step of position k = D - dim
        float d[N];
        uint32_t step[N], base = 0u;
        int s = 0;
#pragma unroll
        for (int dim = 0; dim < N; ++dim) {
            const float e = elevated[dim];
            int q;                           // -q where N is a power of two
            if constexpr (kPow2) {
                // the nearest integer, the lower one in the middle (:98-104 picks up only if it is nearer)
                q = -nearestLower(e);
                d[D - dim] = e + (float)q;
            } else {
                const float down = __builtin_floorf(e * (1.0f / (float)N));
                const bool upper = __builtin_fmaf(down, -(float)N, e) > 0.5f * (float)N;
                const float nearest = upper ? down + 1.0f : down;
                d[D - dim] = __builtin_fmaf(nearest, -(float)N, e);
                q = (int)nearest;
            }
            s += q;
            const uint32_t perUnit = (uint32_t)N * h.mult[dim] - h.all, m = kPow2 ? 0u - perUnit : perUnit;      // N * key, less s * all
            base += ((uint32_t)q & 0xffffffu) * (m & 0xffffffu);
            step[D - dim] = h.all - (uint32_t)N * h.mult[dim];
        }
        if constexpr (kPow2) s = -s;
#pragma unroll
        for (int x = 0; x < kExchanges; ++x) {
            const int k = exchangeAt(x), j = k + apart(x);
            const float a = d[k], b = d[j];
            const uint32_t sa = step[k], sb = step[j];
            bool c = b < a;
            if (N == 4 && x == 4) c = c | ((exchanged[2] | exchanged[3]) & (b <= a));
            exchanged[x] = c;
            d[k] = c ? b : a; d[j] = c ? a : b;
            step[k] = c ? sb : sa; step[j] = c ? sa : sb;
        }
        uint32_t ring[N];
        ring[0] = base;
#pragma unroll
        for (int k = 1; k < N; ++k) ring[k] = ring[k - 1] + step[k - 1];

        const uint32_t by = kPow2 ? (uint32_t)s : (uint32_t)(s < 0 ? s + N : s);
#pragma unroll
        for (int i = 0; i < kTurnBits; ++i) turn[i] = lanesOf((by & (1u << i)) != 0u);
        turnBy(ring, turn);
#pragma unroll
        for (int k = 0; k < N; ++k) hash[k] = ring[k];
        turnBy(d, turn);
        // ranks below `turn` have passed the end (s > 0: rem0 less N), or the others have passed the start (s < 0: rem0 plus N)
        const float unit = kPow2 ? 1.0f : (float)N, others = s < 0 ? -unit : 0.0f, passed = others + unit;
#pragma unroll
        for (int k = 0; k < N; ++k) {
            bool below = false;              // D - k < by
            if constexpr (N <= 4) {
                const Lanes one = turn[0], high = turn[kTurnBits - 1];
                if (k > 0) below = in(D - k == 0 ? one | high : D - k == 1 ? high : one & high);
            } else {
                below = (uint32_t)(D - k) < by;
            }
            d[k] += below ? passed : others;
            if constexpr (!kPow2) d[k] *= 1.0f / (float)N;
        }
        bary[0] = d[0] + (1.0f - d[D]);
#pragma unroll
        for (int k = 1; k < N; ++k) bary[k] = d[k] - d[k - 1];
    }

    // v rounded to the nearest integer, the lower one in the middle
    static CV_LATTICE_FN int nearestLower(float v)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        // v_cvt_rpi rounds to nearest, the upper one in the middle; compared with the other branch for every float below 2^30
        int n;
        asm("v_cvt_rpi_i32_f32 %0, -%1" : "=v"(n) : "v"(v));
        return -n;
#else
        const float near = std::nearbyintf(v);
        return (int)near - (v - near == -0.5f ? 1 : 0);
#endif
    }

    // gradients of the elevated coordinates from those of the weights
    CV_LATTICE_FN void toElevated(const float (&dbary)[N], float (&delev)[N]) const
    {
        float g[N];
#pragma unroll
        for (int k = 0; k < N; ++k) g[k] = (dbary[k] - dbary[(k + 1) % N]) * (1.0f / (float)N);
        turnBack(g, turn);
#pragma unroll
        for (int x = kExchanges - 1; x >= 0; --x) {
            const int k = exchangeAt(x), j = k + apart(x);
            const float a = g[k], b = g[j];
            const bool c = exchanged[x];
            g[k] = c ? b : a; g[j] = c ? a : b;
        }
#pragma unroll
        for (int dim = 0; dim < N; ++dim) delev[dim] = g[D - dim];
    }
};

} // namespace cv
