// cv_train_round.h -- the training step layer by layer inside a workgroup, for networks of half or float of any layer sizes
// that fit its LDS.
//
// The same step as cv_train_general.hip (the example's learnGradient, kernels.slang:9-27, fflayer.slang:29-58; same
// rounding points), but layer by layer over a round of 64 samples in the LDS of one compute unit instead of over the whole
// batch in memory: a workgroup keeps the weights of all layers in LDS, takes its rounds one after the other, and only the
// network's inputs, the targets and one partial of the gradients per workgroup touch memory.
//
// Layout.  Everything is row-major in LDS: W_l as [out][in], the vectors X_l of the round as [64 samples][features], rows
// padded by 16 bytes (which spreads the 16 rows of an operand over all banks).  An MFMA operand whose k axis is the
// feature is read along a row, one whose k axis is the row (W^T in dX = W^T dZ, and both operands of dW = sum_s dZ (x) X)
// down the columns: four 4-byte reads for float, two ds_read_b64_tr_b16 for half.  So one copy of W serves both
// directions and no vector is stored twice: dZ_l takes the place of X_l once dW of the layer above and act'(Z_l) have used
// it.  The sign of a stored activation carries what act' needs: positive where z > 0, +0 at z == 0 (the tie of max()),
// negative or -0 where z < 0 and, behind a ReLU, where z is NaN (which then passes no gradient).
//
// Work split.  Eight waves.  Forward and dX: a wave takes output tiles of 16 features x 16 samples; the epilogue (bias,
// activation, act') is elementwise on its own tiles.  dW: a wave owns tiles of every layer's dW for the whole kernel (in
// registers), contracted over the round's 64 samples; narrow networks also split the samples between waves.  The
// workgroup meets at a barrier between layers, 3 L times per round; two workgroups share a compute unit where LDS and
// registers allow, so that one works while the other meets.
//
// What bounds it: float: the matrix pipeline (v_mfma_f32_16x16x4_f32 takes 32 cycles for what two 4-byte reads supply).
// half: waiting, for operands from LDS (one 16-byte read per lane and operand feeds 16 cycles of the pipeline) and at the
// meetings.  Five float layers up to 64 wide spill 100 registers (196 bytes a lane; 16-64-64-64-64-2 over 2^17 samples 159 us, and
// 169 us with 38 of them while the weights were staged element by element), five half layers beyond 64 wide 13 (44 bytes).
// 16-128-128-128-8 (half) over 200 003 samples: 151 us, 724 us over the whole batch in memory.  187 us while the weights were staged
// element by element (now in 16-byte pieces, all layers requested together) and half networks wider than 64 kept part of the
// prefetched input in scratch memory, so that each round began with a wait for memory.
#pragma once
#include "cv_train_impl.h"

namespace cv {
namespace {

constexpr int kRoundSamples = 64;
// Networks of half wider than 64 whose weights leave no room for the vectors of 64 samples (8-128-128-128-128-4: 123 of 160 KB) take 32 to a
// round: the same tiles of dW, and one row tile of the forward pass and of dX per wave instead of two.  A whole step, over the whole batch in
// memory / in rounds of 32 (us): 8-128-128-128-128-4 over 1 024 samples 165 / 34, over 200 003 943 / 274; 128-128-128-128-9 146 / 30, 798 / 226.
constexpr int kRoundFewSamples = 32;
constexpr int kRoundThreads = 512;
constexpr int kRoundMaxLayers = 5;

struct RoundLayer {
    const uint8_t* w; const uint8_t* bias;
    MatrixShape shape;
    int32_t in, out, act;
    float slope;
    int32_t rowTiles, colTiles;      // 16-feature tiles of the output and of the input
    int32_t kIn, kOut;               // k chunks of the forward pass and of dX
    uint32_t wOff, wStride;          // bytes in LDS: W, and from one of its rows to the next
    uint32_t biasOff;
    uint32_t xOff, xStride;          // the layer's input vectors (dZ of the layer below after its turn)
    uint32_t tileBase, dbBase;       // in the partial: first dW tile, first group of 16 bias gradients
};
struct RoundArgs {
    RoundLayer layers[kRoundMaxLayers];      // (first: the kernel finds them at the head of its arguments)
    uint32_t zOff, zStride;          // dZ of the last layer
    uint32_t ldsBytes;               // the last 16 of them: the workgroup's largest per-sample loss
    const uint8_t* in; uint64_t inStride;
    const uint8_t* targets; uint64_t targetStride;
    uint32_t batch;
    uint32_t samples;                // of a round
    int32_t inPieces;                // input rows of whole aligned 16-byte pieces: their number, else 0
    float lossScale;
    float* partials;
    uint32_t partialFloats, dwTiles; // of a partial: all floats, and the dW tiles ahead of the bias gradients
    int32_t wantLossMax;
    TrainReduceArgs finish;
};

// Tiles per wave.  RT: half the 16-feature tiles of the widest layer, rounded up to 4 or 8 (RT = 2, 4).
template <int RT, int SAMPLES>
struct RoundSplit {
    // forward and dX: NS sample tiles x NT row tiles per wave; the waves of a sample group take every RG-th row tile
    static constexpr int NS = RT == 4 ? 2 : 1, SG = SAMPLES / 16 / NS, RG = 8 / SG, NT = SAMPLES / 32;
    // dW: WR x WC waves tile the matrix, KS of them the samples; RI x CJ tiles per wave
    static constexpr int WR = RT == 4 ? 4 : 2, WC = 2, KS = RT == 4 ? 1 : 2;
    static constexpr int RI = 2, CJ = RT == 2 ? 2 : 4;
    static constexpr int kMaxTiles = 2 * RT;
    static_assert(RG * NT >= kMaxTiles && WR * RI >= kMaxTiles && WC * CJ >= kMaxTiles && WR * WC * KS == 8, "every tile has a wave");
};

// The element types: how operands are read from LDS and multiplied.  A chunk is KC values of the k axis.
template <typename T> struct RoundMma;
template <> struct RoundMma<float> {
    static constexpr int KC = 16;
    typedef floatx4 Op;
    // k along a row: lane group g holds k = 4g .. 4g+3 of the chunk, in both operands of a product
    static __device__ __forceinline__ Op readRow(const uint8_t* row, int g) { return *(const floatx4*)(row + 16 * g); }
    static __device__ __forceinline__ Op readRowSplit(const uint8_t* row, int g) { return readRow(row, g); }
    // k down the rows: lane 16g + i holds column i of rows 4g .. 4g+3 (`p`: the chunk's first row, the tile's first column)
    static __device__ __forceinline__ Op readColumn(const uint8_t* p, uint32_t stride, int g, int i)
    {
        const uint8_t* q = p + (uint32_t)(4 * g) * stride + 4 * i;
        return Op{*(const float*)q, *(const float*)(q + stride), *(const float*)(q + 2 * stride), *(const float*)(q + 3 * stride)};
    }
    // the same of a matrix of sixteen rows (which a chunk has)
    static __device__ __forceinline__ Op readColumnOf16(const uint8_t* p, uint32_t stride, int g, int i) { return readColumn(p, stride, g, i); }
    static __device__ __forceinline__ floatx4 mma(Op a, Op b, floatx4 c)
    {
#pragma unroll
        for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
        return c;
    }
    static __device__ __forceinline__ float sum(Op a, float s) { return s + ((a[0] + a[1]) + (a[2] + a[3])); }
    // z -> stored activation (see the head of this file), four at a time
    static __device__ __forceinline__ void storeActivated(uint8_t* p, floatx4 z, int act, float slope)
    {
        if (act == kActRelu) {
#pragma unroll
            for (int r = 0; r < 4; ++r) z[r] = z[r] > 0.f ? z[r] : (z[r] == 0.f ? 0.f : -0.f);      // (NaN: -0)
        } else if (act == kActLeakyRelu) {
#pragma unroll
            for (int r = 0; r < 4; ++r) { const float u = z[r] + 0.f; z[r] = fmaxf(u, u * slope); }      // (-0 + 0 = +0)
        }
        *(floatx4*)p = z;
    }
    static __device__ __forceinline__ bool isPlusZero(float v) { return __builtin_bit_cast(uint32_t, v) == 0u; }
    // dz = g * act'(z), from the stored activation at p, in its place
    static __device__ __forceinline__ floatx4 storeGradient(uint8_t* p, floatx4 g, int act, float slope)
    {
        if (act == kActRelu) {
            const floatx4 x = *(const floatx4*)p;
#pragma unroll
            for (int r = 0; r < 4; ++r) g[r] = x[r] > 0.f ? g[r] : (isPlusZero(x[r]) ? 0.5f * g[r] : 0.f);
        } else if (act == kActLeakyRelu) {
            const floatx4 x = *(const floatx4*)p;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float half = 0.5f * g[r];
                g[r] = x[r] > 0.f ? g[r] : (isPlusZero(x[r]) ? half + half * slope : g[r] * slope);
            }
        }
        *(floatx4*)p = g;
        return g;
    }
};
template <> struct RoundMma<half_t> {
    static constexpr int KC = 32;
    typedef u32x4 Op;
    static __device__ __forceinline__ Op readRow(const uint8_t* row, int g) { return *(const u32x4*)(row + 16 * g); }
    // with the k order of readColumn: 4g .. 4g+3, then 16+4g .. 16+4g+3
    static __device__ __forceinline__ Op readRowSplit(const uint8_t* row, int g)
    {
        const u32x2 lo = *(const u32x2*)(row + 8 * g), hi = *(const u32x2*)(row + 32 + 8 * g);
        return Op{lo.x, lo.y, hi.x, hi.y};
    }
    // lane 16g + i receives column i of rows 4g .. 4g+3 and 16+4g .. 16+4g+3: within a 16-lane group lane q hands in the
    // address of four halves of row 4g + q/4 (see readF in cv_train_pair.h for what the instruction returns)
    static __device__ __forceinline__ Op readColumn(const uint8_t* p, uint32_t stride, int g, int i)
    {
        typedef short shortx4 __attribute__((ext_vector_type(4)));
        typedef shortx4 __attribute__((address_space(3))) * LdsPtr;
        const uint8_t* q = p + (uint32_t)(4 * g + (i >> 2)) * stride + 8 * (i & 3);
        const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsPtr)q));
        const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsPtr)(q + 16 * stride)));
        return Op{lo.x, lo.y, hi.x, hi.y};
    }
    // the same of a matrix of sixteen rows
    static __device__ __forceinline__ Op readColumnOf16(const uint8_t* p, uint32_t stride, int g, int i)
    {
        typedef short shortx4 __attribute__((ext_vector_type(4)));
        typedef shortx4 __attribute__((address_space(3))) * LdsPtr;
        const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsPtr)(p + (uint32_t)(4 * g + (i >> 2)) * stride + 8 * (i & 3))));
        return Op{lo.x, lo.y, 0u, 0u};
    }
    static __device__ __forceinline__ floatx4 mma(Op a, Op b, floatx4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(halfx8, a), __builtin_bit_cast(halfx8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ float sum(Op a, float s)
    {
        const halfx2 ones = {(half_t)1.f, (half_t)1.f};
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const uint32_t pair = a[d];      // (a variable of its own: __builtin_bit_cast of a vector's element takes element 0)
            s = __builtin_amdgcn_fdot2(__builtin_bit_cast(halfx2, pair), ones, s, false);
        }
        return s;
    }
    static __device__ __forceinline__ halfx2 round2(float a, float b)
    {
        typedef float floatx2 __attribute__((ext_vector_type(2)));
        return __builtin_convertvector(floatx2{a, b}, halfx2);
    }
    static __device__ __forceinline__ void storeActivated(uint8_t* p, floatx4 acc, int act, float slope)
    {
        const halfx2 zero = {(half_t)0, (half_t)0};
        const halfx2 z0 = round2(acc[0], acc[1]) + zero, z1 = round2(acc[2], acc[3]) + zero;      // (-0 + 0 = +0)
        u32x2 x = {__builtin_bit_cast(uint32_t, z0), __builtin_bit_cast(uint32_t, z1)};
        if (act == kActRelu) {      // (a NaN leaves the matrix instruction with its sign set, whatever it came from: -0)
            x.x = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(z0, zero)) | (x.x & 0x80008000u);
            x.y = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(z1, zero)) | (x.y & 0x80008000u);
        } else if (act == kActLeakyRelu) {
            const half_t sl = (half_t)slope;
            const halfx2 s2 = {sl, sl};
            x.x = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(z0, z0 * s2));
            x.y = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(z1, z1 * s2));
        }
        *(u32x2*)p = x;
    }
    // {1, 0.5, 0} for a positive, zero, negative stored activation: as 16-bit integers the three kinds are > 0, 0 and below
    // -14, so clamped to [-14, 1] and taken times 1024 plus 0x3800 they become the bits of those halfs
    static __device__ __forceinline__ halfx2 multiplier(uint32_t x)
    {
        typedef short shortx2 __attribute__((ext_vector_type(2)));
        const shortx2 v = __builtin_elementwise_max(__builtin_elementwise_min(__builtin_bit_cast(shortx2, x), shortx2{1, 1}), shortx2{-14, -14});
        return __builtin_bit_cast(halfx2, (shortx2)(v * shortx2{1024, 1024} + shortx2{0x3800, 0x3800}));
    }
    static __device__ __forceinline__ void storeGradient(uint8_t* p, floatx4 g, int act, float slope)
    {
        halfx2 d0 = round2(g[0], g[1]), d1 = round2(g[2], g[3]);
        if (act == kActRelu) {
            const u32x2 x = *(const u32x2*)p;
            d0 = d0 * multiplier(x.x);
            d1 = d1 * multiplier(x.y);
        } else if (act == kActLeakyRelu) {
            const half_t sl = (half_t)slope;
            const u32x2 x = *(const u32x2*)p;
            d0 = applyActGrad<true>(d0, multiplier(x.x), kActLeakyRelu, halfx2{sl, sl});
            d1 = applyActGrad<true>(d1, multiplier(x.y), kActLeakyRelu, halfx2{sl, sl});
        }
        *(u32x2*)p = u32x2{__builtin_bit_cast(uint32_t, d0), __builtin_bit_cast(uint32_t, d1)};
    }
};

// every wave of the workgroup has finished its LDS accesses; loads from memory stay in flight
__device__ __forceinline__ void meetInLds() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Weights and biases of all layers to LDS.  A row-major matrix (what a program's own matrices mostly are) goes in 16-byte pieces, of
// half at whatever element they begin, and the first kAhead pieces of a thread of every layer are requested before the first is stored:
// one round trip to memory for all of them instead of one for every four elements.  16-128-128-128-8 (half), 64 samples to a workgroup, see
// the head of this file.  Rows of half that are no whole aligned pieces, element by element / so (us): 7-67-16-67-123-1 over 5 923 samples
// 35 / 24, 26-81-11-80-2 over 15 796 24.5 / 20, 12-128-128-128-15 over 1 819 26 / 23.  That is an instantiation of its own (ANY): the longer
// code costs a network that does not need it 1 to 2 us (16-128-128-128-8 over 200 003 samples 151.7 / 154.2), and one of float whose rows do
// (36-64-64-64-64-14 over 3 167 30.6 / 32.1), so that float stays element by element.
template <typename T>
__host__ __device__ __forceinline__ size_t roundWeightLine(const RoundLayer& ly) { return ly.shape.stride ? ly.shape.stride : (size_t)ly.shape.cols * sizeof(T); }
template <typename T>
__device__ __forceinline__ size_t roundWeightBytes(const RoundLayer& ly) { return (size_t)(ly.out - 1) * roundWeightLine<T>(ly) + (size_t)ly.in * sizeof(T); }
// rows of whole aligned pieces
template <typename T>
__host__ __device__ __forceinline__ bool roundWeightWhole(const RoundLayer& ly)
{
    return ((size_t)ly.in * sizeof(T)) % 16u == 0 && (((uintptr_t)ly.w | roundWeightLine<T>(ly)) & 15u) == 0;
}
template <typename T, bool ANY>
__device__ __forceinline__ bool roundWeightPieces(const RoundLayer& ly)
{
    return ly.shape.layout == kRowMajor && (ANY ? roundWeightBytes<T>(ly) >= 16u : roundWeightWhole<T>(ly));
}
template <typename T, int NL, int MAXT, bool ANY = false>
__device__ __forceinline__ void stageRoundWeights(const RoundLayer (&layers)[kRoundMaxLayers], uint8_t* lds)
{
    constexpr int kMost = MAXT * 16 * MAXT * 16 * (int)sizeof(T) / 16 / kRoundThreads, kUpTo = NL < 5 ? 4 : 2, kAhead = kMost < 1 ? 1 : kMost < kUpTo ? kMost : kUpTo;
    u32x4 v[NL][kAhead];
    auto piece = [&](const RoundLayer& ly, uint32_t c, uint32_t& row, uint32_t& at) {
        const uint32_t perRow = ((uint32_t)ly.in * sizeof(T) + 15u) / 16u;
        row = c / perRow;
        at = c - row * perRow;
        return row < (uint32_t)ly.out;
    };
    // (a piece that would end behind the matrix is read ending there and moved down; what lies behind its row is cleared)
    auto load = [&](const RoundLayer& ly, bool whole, uint32_t row, uint32_t at) {
        if (whole) return *(const u32x4*)(ly.w + row * roundWeightLine<T>(ly) + 16u * at);
        const size_t off = row * roundWeightLine<T>(ly) + 16u * at, last = roundWeightBytes<T>(ly) - 16u;
        return ((const Loose16<(int)sizeof(T)>*)(ly.w + (off < last ? off : last)))->v;
    };
    auto store = [&](const RoundLayer& ly, bool whole, uint32_t row, uint32_t at, u32x4 v) {
        if (!whole) {
            const size_t off = row * roundWeightLine<T>(ly) + 16u * at, last = roundWeightBytes<T>(ly) - 16u;
            uint32_t x[4] = {v.x, v.y, v.z, v.w};
            if (off > last) shiftDown<(int)sizeof(T)>(x, (int)(off - last));
            clearBehind<(int)sizeof(T)>(x, ly.in * (int)sizeof(T) - 16 * (int)at);
            v = u32x4{x[0], x[1], x[2], x[3]};
        }
        *(u32x4*)(lds + ly.wOff + row * ly.wStride + 16u * at) = v;
    };
    float bias[NL];
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        const RoundLayer& ly = layers[l];
        const int e = threadIdx.x;
        bias[l] = ly.bias && e < ly.out ? (float)((const T*)ly.bias)[e] : 0.f;      // (no layer has more rows than the workgroup threads)
        if (!roundWeightPieces<T, ANY>(ly)) continue;
        const bool whole = !ANY || roundWeightWhole<T>(ly);
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            uint32_t row, at;
            const bool on = piece(ly, threadIdx.x + (uint32_t)(i * kRoundThreads), row, at);
            v[l][i] = load(ly, whole, on ? row : 0u, on ? at : 0u);
        }
    }
#pragma unroll
    for (int l = 0; l < NL; ++l) {
        const RoundLayer& ly = layers[l];
        if ((int)threadIdx.x < ly.out) *(float*)(lds + ly.biasOff + 4 * threadIdx.x) = bias[l];
        uint32_t row, at;
        if (roundWeightPieces<T, ANY>(ly)) {
            const bool whole = !ANY || roundWeightWhole<T>(ly);
#pragma unroll
            for (int i = 0; i < kAhead; ++i)
                if (piece(ly, threadIdx.x + (uint32_t)(i * kRoundThreads), row, at)) store(ly, whole, row, at, v[l][i]);
            for (uint32_t c = threadIdx.x + (uint32_t)(kAhead * kRoundThreads); piece(ly, c, row, at); c += kRoundThreads) store(ly, whole, row, at, load(ly, whole, row, at));
        } else {
            const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
            for (int col = lane; col < ly.in; col += 64) {
#pragma unroll 4
                for (int r = wave; r < ly.out; r += kRoundThreads / 64)
                    *(T*)(lds + ly.wOff + (uint32_t)r * ly.wStride + (uint32_t)col * sizeof(T)) = *(const T*)(ly.w + elemOffset(ly.shape, (uint32_t)r, (uint32_t)col));
            }
        }
    }
}

// WAVES: per SIMD; 4 where two workgroups share a compute unit (128 registers a wave), else 2
// ANY (half): some matrix is row-major with rows that are no whole aligned pieces
template <typename T, int NL, int RT, int WAVES, int SAMPLES, bool ANY>
__global__ __launch_bounds__(kRoundThreads) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES))) void trainRoundKernel(const RoundArgs a)
{
    typedef RoundMma<T> M;
    typedef RoundSplit<RT, SAMPLES> S;
    typedef typename M::Op Op;
    constexpr int KC = M::KC, ESZ = sizeof(T), NS = S::NS, NT = S::NT;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    uint32_t* const ldsLossMax = (uint32_t*)(lds + a.ldsBytes - 16);

    for (uint32_t i = threadIdx.x; i < a.ldsBytes / 16; i += kRoundThreads) ((u32x4*)lds)[i] = u32x4{0u, 0u, 0u, 0u};
    __syncthreads();
    stageRoundWeights<T, NL, 2 * RT, ANY>(a.layers, lds);
    __syncthreads();

    // The layers' sizes and places in LDS are read from the kernel's arguments where they are used (scalar loads): hoisted out
    // of the rounds, as they would be, they and the addresses made of them take more registers than a wave has.
    typedef const RoundLayer __attribute__((address_space(4))) LayerInArgs;
    auto layer = [](int l) -> LayerInArgs& {
        LayerInArgs* p = (LayerInArgs*)__builtin_amdgcn_kernarg_segment_ptr() + l;
        asm volatile("" : "+s"(p));
        return *p;
    };
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sg = wave % S::SG, rg = wave / S::SG;                                       // forward and dX
    const int wc = wave % S::WC, ks = wave / S::WC % S::KS, wr = wave / (S::WC * S::KS);    // dW

    floatx4 accW[NL][S::RI][S::CJ];
    float accB[NL][S::RI];
#pragma unroll
    for (int l = 0; l < NL; ++l)
#pragma unroll
        for (int i = 0; i < S::RI; ++i) {
            accB[l][i] = 0.f;
#pragma unroll
            for (int j = 0; j < S::CJ; ++j) accW[l][i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
        }
    float lossAcc = 0.f, lossMaxAcc = 0.f;

    const uint32_t lastSample = a.batch - 1, numRounds = lastSample / SAMPLES + 1;

    // ---- the network's input: eight threads (sixteen) to a sample, 16-byte pieces where rows are made of them, else elements.
    //      Addresses always exist; what lies past the vector is not stored.
    constexpr int PER = kRoundThreads / SAMPLES, PIECES = (2 * RT * 16 * ESZ / 16 + PER - 1) / PER, ELEMS = 2 * RT * 16 / PER;
    constexpr int IN_REGS = 4 * PIECES > ELEMS ? 4 * PIECES : ELEMS;
    const int inRow = threadIdx.x / PER;
    const int in0 = a.layers[0].in, topOut = a.layers[NL - 1].out;
    auto fetchInput = [&](uint32_t (&v)[IN_REGS], uint32_t r) {
        int inCol = threadIdx.x % PER;
        pinHere(inCol);                     // (the addresses are formed anew each round, see layer())
        const uint8_t* row = a.in + (size_t)min(r * SAMPLES + inRow, lastSample) * a.inStride;
        if (a.inPieces) {
#pragma unroll
            for (int c = 0; c < PIECES; ++c) {
                const u32x4 p = *(const u32x4*)(row + 16 * min(inCol + PER * c, a.inPieces - 1));
                v[4 * c] = p.x; v[4 * c + 1] = p.y; v[4 * c + 2] = p.z; v[4 * c + 3] = p.w;
            }
            asm volatile("");               // (the ends of the two branches differ: else their stores become one, to an address
                                            // chosen between registers, and the array moves to scratch memory)
        } else {
#pragma unroll
            for (int c = 0; c < ELEMS; ++c) {
                const uint8_t* p = row + ESZ * min(inCol + PER * c, in0 - 1);
                v[c] = ESZ == 4 ? *(const uint32_t*)p : *(const uint16_t*)p;
            }
        }
    };
    auto putInput = [&](const uint32_t (&v)[IN_REGS]) {
        int inCol = threadIdx.x % PER;
        pinHere(inCol);
        LayerInArgs& ly = layer(0);
        uint8_t* row = lds + ly.xOff + (uint32_t)inRow * ly.xStride;
        if (a.inPieces) {
#pragma unroll
            for (int c = 0; c < PIECES; ++c)
                if (inCol + PER * c < a.inPieces) *(u32x4*)(row + 16 * (inCol + PER * c)) = u32x4{v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]};
        } else {
#pragma unroll
            for (int c = 0; c < ELEMS; ++c)
                if (inCol + PER * c < in0) {
                    if constexpr (ESZ == 4) *(uint32_t*)(row + 4 * (inCol + PER * c)) = v[c];
                    else *(uint16_t*)(row + 2 * (inCol + PER * c)) = (uint16_t)v[c];
                }
        }
    };

    // ---- forward: `count` of this wave's row tiles of layer l, times its sample tiles -----------------------------------
    auto product = [&](auto countC, LayerInArgs& ly, floatx4 (&acc)[NS][NT]) {
        constexpr int count = decltype(countC)::value;
        const uint8_t* w = lds + ly.wOff + (uint32_t)(16 * rg + n) * ly.wStride;
        const uint8_t* x = lds + ly.xOff + (uint32_t)(16 * NS * sg + n) * ly.xStride;
#pragma unroll
        for (int t = 0; t < count; ++t) {
            const floatx4 b = *(const floatx4*)(lds + ly.biasOff + 4 * (16 * (rg + S::RG * t) + 4 * g));
#pragma unroll
            for (int s = 0; s < NS; ++s) acc[s][t] = b;
        }
#pragma unroll 2
        for (int k = 0; k < ly.kIn; ++k) {
            Op av[count], bv[NS];
#pragma unroll
            for (int t = 0; t < count; ++t) av[t] = M::readRow(w + (uint32_t)(16 * S::RG * t) * ly.wStride + k * KC * ESZ, g);
#pragma unroll
            for (int s = 0; s < NS; ++s) bv[s] = M::readRow(x + (uint32_t)(16 * s) * ly.xStride + k * KC * ESZ, g);
#pragma unroll
            for (int t = 0; t < count; ++t)
#pragma unroll
                for (int s = 0; s < NS; ++s) acc[s][t] = M::mma(av[t], bv[s], acc[s][t]);
        }
    };
    auto forward = [&](auto countC, LayerInArgs& ly, uint32_t outOff, uint32_t outStride) {
        constexpr int count = decltype(countC)::value;
        floatx4 acc[NS][NT];
        product(countC, ly, acc);
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int t = 0; t < count; ++t)
                M::storeActivated(lds + outOff + (uint32_t)(16 * (NS * sg + s) + n) * outStride + (16 * (rg + S::RG * t) + 4 * g) * ESZ, acc[s][t], ly.act, ly.slope);
    };

    // ---- dW and db of layer l over this wave's samples of the round ------------------------------------------------------
    auto contract = [&](auto lc, auto rowsC, auto colsC, uint32_t dzOff, uint32_t dzStride) {
        constexpr int l = decltype(lc)::value, rows = decltype(rowsC)::value, cols = decltype(colsC)::value;
        constexpr int chunks = SAMPLES / S::KS / KC;
        LayerInArgs& ly = layer(l);
        const uint8_t* dz = lds + dzOff + 16 * wr * ESZ;
        const uint8_t* x = lds + ly.xOff + 16 * wc * ESZ;
#pragma unroll
        for (int c = 0; c < chunks; ++c) {
            const uint32_t row = (uint32_t)((ks * chunks + c) * KC);
            Op av[rows], bv[cols];
#pragma unroll
            for (int i = 0; i < rows; ++i) av[i] = M::readColumn(dz + row * dzStride + 16 * S::WR * i * ESZ, dzStride, g, n);
#pragma unroll
            for (int j = 0; j < cols; ++j) bv[j] = M::readColumn(x + row * ly.xStride + 16 * S::WC * j * ESZ, ly.xStride, g, n);
#pragma unroll
            for (int i = 0; i < rows; ++i) {
#pragma unroll
                for (int j = 0; j < cols; ++j) accW[l][i][j] = M::mma(av[i], bv[j], accW[l][i][j]);
                if (wc == 0) accB[l][i] = M::sum(av[i], accB[l][i]);
            }
        }
    };
    // how many of `tiles` tiles, dealt to `step` waves, wave `at` has
    auto share = [](int tiles, int at, int step) { return tiles > at ? (tiles - at + step - 1) / step : 0; };

    auto targetValue = [](uint32_t bits) -> float {
        if constexpr (ESZ == 4) return __builtin_bit_cast(float, bits);
        else return (float)__builtin_bit_cast(half_t, (uint16_t)bits);
    };

    // ---- rounds ----------------------------------------------------------------------------------------------------------
    uint32_t nextIn[IN_REGS];
    fetchInput(nextIn, blockIdx.x);
    for (uint32_t r = blockIdx.x; r < numRounds; r += gridDim.x) {
        putInput(nextIn);
        meetInLds();
        fetchInput(nextIn, r + gridDim.x);
        // targets of the waves that will form the loss
        uint32_t tgt[NS][4];
        if (rg == 0 && a.targets) {
            int g4 = 4 * g;
            pinHere(g4);
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                {
                    const uint8_t* p = a.targets + (size_t)min(r * SAMPLES + 16 * (NS * sg + s) + n, lastSample) * a.targetStride + ESZ * min(g4 + q, topOut - 1);
                    tgt[s][q] = ESZ == 4 ? *(const uint32_t*)p : *(const uint16_t*)p;
                }
        }
        asm volatile("" ::: "memory");      // the requests stay here

        for (int l = 0; l + 1 < NL; ++l) {
            LayerInArgs& ly = layer(l);
            LayerInArgs& next = layer(l + 1);
            const int mine = share(ly.rowTiles, rg, S::RG);
            if (mine == 2) forward(std::integral_constant<int, NT>{}, ly, next.xOff, next.xStride);
            else if (mine) forward(std::integral_constant<int, 1>{}, ly, next.xOff, next.xStride);
            meetInLds();
        }
        // the last layer has one row tile: loss and its gradient at the pre-activations
        if (rg == 0) {
            LayerInArgs& top = layer(NL - 1);
            floatx4 acc[NS][NT];
            product(std::integral_constant<int, 1>{}, top, acc);
            // (the sample tile a constant from the start: an array indexed by a loop that is unrolled too late lies in scratch
            // memory, and its loads wait for the prefetched input as well)
            staticFor<0, NS>([&](auto sc) {
                constexpr int s = decltype(sc)::value;
                const int row = 16 * (NS * sg + s) + n;
                const bool live = r * SAMPLES + row < a.batch;
                float tgtAll = 0.f;
                if (!a.targets) {
                    // sin(sum of the inputs), each lane group a quarter of them, as the other steps form it
                    const int gs = (int)optGS((uint32_t)in0);
                    LayerInArgs& first = layer(0);
                    const T* xin = (const T*)(lds + first.xOff + (uint32_t)row * first.xStride);
                    float part = 0.f;
                    for (int q = 0; q < gs; ++q) part += g * gs + q < in0 ? (float)xin[g * gs + q] : 0.f;
                    tgtAll = (float)(T)sinf(sumOverGroups(part));
                }
                float sampleLoss = 0.f;
                T dz[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const bool on = live && 4 * g + q < top.out;
                    const T z = (T)acc[s][0][q];
                    const float zs = (float)(T)((float)z * (float)(T)top.slope);
                    float y = (float)z;
                    if (top.act == kActRelu) y = y > 0.f ? y : 0.f;
                    if (top.act == kActLeakyRelu) y = fmaxf(y, zs);
                    const T diff = (T)(y - (a.targets ? targetValue(tgt[s][q]) : tgtAll));
                    sampleLoss += on ? (float)diff * (float)diff : 0.f;
                    const T gv = (T)(2.0f * (float)diff * a.lossScale), hg = (T)(0.5f * (float)gv);
                    T d = gv;
                    if (top.act == kActRelu) d = (float)z > 0.f ? gv : ((float)z == 0.f ? hg : (T)0.f);
                    if (top.act == kActLeakyRelu) {
                        const T da = (float)z > 0.f ? gv : ((float)z == 0.f ? hg : (T)0.f), db = (float)z > 0.f ? (T)0.f : ((float)z == 0.f ? hg : gv);
                        d = (T)((float)da + (float)(T)((float)db * (float)(T)top.slope));
                    }
                    dz[q] = on ? d : (T)0.f;
                }
                lossAcc += sampleLoss;
                if (a.wantLossMax) {
                    const float whole = sumOverGroups(sampleLoss);
                    lossMaxAcc = (whole > lossMaxAcc || whole != whole) ? whole : lossMaxAcc;
                }
                T* out = (T*)(lds + a.zOff + (uint32_t)row * a.zStride + 4 * g * ESZ);
                typedef T TVec __attribute__((ext_vector_type(4)));
                *(TVec*)out = TVec{dz[0], dz[1], dz[2], dz[3]};
            });
        }
        meetInLds();

        staticFor<0, NL>([&](auto ic) {
            constexpr int l = NL - 1 - decltype(ic)::value;
            typedef std::integral_constant<int, l> LC;
            LayerInArgs& ly = layer(l);
            LayerInArgs& above = layer(l + 1 < NL ? l + 1 : l);
            const uint32_t dzOff = l + 1 < NL ? above.xOff : a.zOff, dzStride = l + 1 < NL ? above.xStride : a.zStride;
            const int rows = share(ly.rowTiles, wr, S::WR), cols = share(ly.colTiles, wc, S::WC);
            staticFor<1, S::RI + 1>([&](auto rc) {
                staticFor<1, S::CJ + 1>([&](auto cc) {
                    if (rows == decltype(rc)::value && cols == decltype(cc)::value) contract(LC{}, rc, cc, dzOff, dzStride);
                });
            });
            if constexpr (l > 0) {
                // dX = W^T dZ on the wave's tiles of the layer's input (those beyond it: computed from its last tile, not kept)
                const int mine = share(ly.colTiles, rg, S::RG);
                floatx4 acc[NS][NT];
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[s][t] = floatx4{0.f, 0.f, 0.f, 0.f};
                if (mine) {
                    const uint8_t* dz = lds + dzOff + (uint32_t)(16 * NS * sg + n) * dzStride;
#pragma unroll 2
                    for (int k = 0; k < ly.kOut; ++k) {
                        Op av[NT], bv[NS];
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            const uint8_t* w = lds + ly.wOff + (uint32_t)(k * KC) * ly.wStride + 16 * (rg + S::RG * (t < mine ? t : 0)) * ESZ;
                            if constexpr (SAMPLES == kRoundFewSamples && l + 1 == NL) av[t] = M::readColumnOf16(w, ly.wStride, g, n);
                            else av[t] = M::readColumn(w, ly.wStride, g, n);
                        }
#pragma unroll
                        for (int s = 0; s < NS; ++s) bv[s] = M::readRowSplit(dz + (uint32_t)(16 * s) * dzStride + k * KC * ESZ, g);
#pragma unroll
                        for (int t = 0; t < NT; ++t)
#pragma unroll
                            for (int s = 0; s < NS; ++s) acc[s][t] = M::mma(av[t], bv[s], acc[s][t]);
                    }
                }
                meetInLds();          // everybody is done with X_l
                LayerInArgs& below = layer(l - 1);
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        if (t < mine)
                            M::storeGradient(lds + ly.xOff + (uint32_t)(16 * (NS * sg + s) + n) * ly.xStride + (16 * (rg + S::RG * t) + 4 * g) * ESZ, acc[s][t],
                                             below.act, below.slope);
            }
            meetInLds();
        });
    }

    // ---- the workgroup's partial: waves that shared tiles by samples are added in a fixed order through LDS ---------------
    __syncthreads();
    float* part = a.partials + (size_t)blockIdx.x * a.partialFloats;
    if (a.wantLossMax) noteLossMax(ldsLossMax, lossMaxAcc);
    float* red = (float*)lds;
    red[threadIdx.x] = lossAcc;
    __syncthreads();
    if (wave == 0) {
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < 8; ++w) s += red[64 * w + lane];
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) s += __shfl_xor(s, d, 64);
        if (lane == 0) {
            part[a.partialFloats - 16] = s;
            part[a.partialFloats - 15] = __builtin_bit_cast(float, *ldsLossMax);
        }
    }
    staticFor<0, NL>([&](auto lc) {
        constexpr int l = decltype(lc)::value;
        LayerInArgs& ly = layer(l);
        const int rows = share(ly.rowTiles, wr, S::WR), cols = share(ly.colTiles, wc, S::WC);
        float* mine = red + (wr * S::WC + wc) * (S::RI * S::CJ * 256);
        float* mineB = red + S::WR * S::WC * S::RI * S::CJ * 256 + wr * (S::RI * 16);
        if constexpr (S::KS > 1) {
            __syncthreads();
            if (ks == 1) {
#pragma unroll
                for (int i = 0; i < S::RI; ++i)
#pragma unroll
                    for (int j = 0; j < S::CJ; ++j) *(floatx4*)&mine[(i * S::CJ + j) * 256 + 4 * lane] = accW[l][i][j];
            }
        }
        // a row's bias gradient lies in the four lane groups
        float b[S::RI];
#pragma unroll
        for (int i = 0; i < S::RI; ++i) {
            b[i] = accB[l][i] + __shfl_xor(accB[l][i], 16, 64);
            b[i] += __shfl_xor(b[i], 32, 64);
            if (S::KS > 1 && ks == 1 && wc == 0 && g == 0) mineB[16 * i + n] = b[i];
        }
        if constexpr (S::KS > 1) __syncthreads();
        if (ks == 0) {
#pragma unroll
            for (int i = 0; i < S::RI; ++i) {
                if (i >= rows) continue;
#pragma unroll
                for (int j = 0; j < S::CJ; ++j) {
                    if (j >= cols) continue;
                    floatx4 v = accW[l][i][j];
                    if constexpr (S::KS > 1) v += *(const floatx4*)&mine[(i * S::CJ + j) * 256 + 4 * lane];
                    const uint32_t tile = ly.tileBase + (uint32_t)((wr + S::WR * i) * ly.colTiles + wc + S::WC * j);
                    __builtin_nontemporal_store(v, (floatx4*)&part[tile * 256 + 4 * lane]);
                }
                if (wc == 0 && g == 0) {
                    if constexpr (S::KS > 1) b[i] += mineB[16 * i + n];
                    part[a.dwTiles * 256 + (ly.dbBase + wr + S::WR * i) * 16 + n] = b[i];
                }
            }
        }
    });
}

// where value p of a summed partial belongs (see gradientSlot): the layers' tiles of 16 x 16, then their bias gradients
__device__ __forceinline__ uint8_t* roundGradientSlot(const RoundArgs& a, int numLayers, uint32_t p)
{
    const TrainReduceArgs& ra = a.finish;
    const uint32_t esz = ra.gradCt == kF32 ? 4u : 2u, nW = a.dwTiles * 256u;
    uint8_t* slot = nullptr;
    for (int l = 0; l < numLayers; ++l) {
        const RoundLayer& ly = a.layers[l];
        const TrainReduceArgs::Layer& dst = ra.layers[l];
        const uint32_t w0 = ly.tileBase * 256u, w1 = w0 + (uint32_t)(ly.rowTiles * ly.colTiles) * 256u;
        const uint32_t b0 = nW + ly.dbBase * 16u, b1 = b0 + (uint32_t)ly.rowTiles * 16u;
        if (p >= w0 && p < w1) {
            const uint32_t q = p - w0, tile = q >> 8, ln = (q >> 2) & 63u;
            const uint32_t o = 16u * (tile / (uint32_t)ly.colTiles) + 4u * (ln >> 4) + (q & 3u), i = 16u * (tile % (uint32_t)ly.colTiles) + (ln & 15u);
            if (dst.wGrad && o < (uint32_t)ly.out && i < (uint32_t)ly.in) slot = dst.wGrad + elemOffset(dst.gradShape, o, i);
        } else if (p >= b0 && p < b1) {
            const uint32_t o = p - b0;
            if (dst.bGrad && o < (uint32_t)ly.out) slot = dst.bGrad + (size_t)o * esz;
        }
    }
    return slot;
}

// Sums the workgroups' partials in a fixed order and adds them to the gradients (mlpTrainReduceKernel for run-time sizes; a
// loss that is not finite voids the step here, too).
__global__ __launch_bounds__(64 * kReduceWaves) void trainRoundReduceKernel(const RoundArgs a)
{
    const TrainReduceArgs& ra = a.finish;
    __shared__ float red[kReduceWaves * 64];
    __shared__ uint32_t maxBits;
    const uint32_t lossAt = a.partialFloats - 16u, p = blockIdx.x * 64u + (threadIdx.x & 63u);
    const bool inRange = p <= lossAt, ownsLoss = blockIdx.x == lossAt / 64u;
    if (threadIdx.x == 0) maxBits = 0u;
    __syncthreads();
    bool voidStep = false;
    for (uint32_t b = threadIdx.x; b < ra.numPartials; b += 64u * kReduceWaves) {
        const float lp = ra.partials[(size_t)b * a.partialFloats + lossAt];
        voidStep = voidStep || notFinite(lp);
        if (ra.lossMax && ownsLoss) atomicMax(&maxBits, __builtin_bit_cast(uint32_t, ra.partials[(size_t)b * a.partialFloats + lossAt + 1u]));
    }
    uint8_t* slot = nullptr;
    float old = 0.f;
    if (threadIdx.x < 64u && p < lossAt) {
        slot = roundGradientSlot(a, ra.numLayers, p);
        if (slot) old = loadGradient(slot, ra.gradCt);
    }
    float s;
    const bool mine = sumPartials(ra.partials + p, a.partialFloats, ra.numPartials, inRange, red, s);
    voidStep = __syncthreads_or(voidStep) != 0;
    if (ra.lossMax && ownsLoss && threadIdx.x == 0) *ra.lossMax = voidStep ? __builtin_nanf("") : __builtin_bit_cast(float, maxBits);
    if (!mine || !inRange) return;
    if (voidStep) s = __builtin_nanf("");
    if (p == lossAt) {
        if (ra.lossSum) *ra.lossSum = s;
        return;
    }
    if (slot) storeGradient(slot, ra.gradCt, old + s);
}

// ---- host side -----------------------------------------------------------------------------------------------------------

// Lays the network out in LDS.  False where the kernel does not apply: more than five layers, more than 128 inputs or hidden
// units, more than 16 outputs, an input encoding, or weights and a round that do not fit the LDS of a compute unit.
inline bool planRoundOf(uint32_t samples, const MlpArgs& m, int ct, RoundArgs& a, int& maxTiles)
{
    const uint32_t esz = elemSize(ct), kc = ct == kF32 ? 16u : 32u;
    const int L = m.numLayers;
    if (L < 2 || L > kRoundMaxLayers || m.inEncoding != kEncodeNone || m.layers[L - 1].out > 16) return false;
    auto up = [](uint32_t v, uint32_t to) { return (v + to - 1u) / to * to; };
    uint32_t off = 0, tiles = 0, groups = 0;
    maxTiles = 1;
    for (int l = 0; l < L; ++l) {
        RoundLayer& ly = a.layers[l];
        const MlpLayerArgs& src = m.layers[l];
        if (src.in > 128 || src.out > 128 || src.act > kActLeakyRelu) return false;
        ly.w = src.w; ly.bias = src.bias; ly.shape = src.shape;
        ly.in = src.in; ly.out = src.out; ly.act = src.act; ly.slope = src.slope;
        ly.rowTiles = (int32_t)optMT((uint32_t)src.out); ly.colTiles = (int32_t)optMT((uint32_t)src.in);
        ly.kIn = (int32_t)(up((uint32_t)src.in, kc) / kc); ly.kOut = (int32_t)(up((uint32_t)src.out, kc) / kc);
        if (ly.colTiles > maxTiles) maxTiles = ly.colTiles;
        ly.wStride = (uint32_t)ly.kIn * kc * esz + 16u;
        ly.wOff = off; off += (samples == (uint32_t)kRoundFewSamples && l + 1 == L ? 16u : (uint32_t)ly.kOut * kc) * ly.wStride;      // (readColumnOf16)
        ly.tileBase = tiles; tiles += (uint32_t)(ly.rowTiles * ly.colTiles);
        ly.dbBase = groups; groups += (uint32_t)ly.rowTiles;
    }
    for (int l = 0; l < L; ++l) { a.layers[l].biasOff = off; off += (uint32_t)a.layers[l].rowTiles * 64u; }
    for (int l = 0; l < L; ++l) {
        a.layers[l].xStride = (uint32_t)a.layers[l].kIn * kc * esz + 16u;
        a.layers[l].xOff = off; off += samples * a.layers[l].xStride;
    }
    a.zStride = (uint32_t)a.layers[L - 1].kOut * kc * esz + 16u;
    a.zOff = off; off += samples * a.zStride;
    constexpr uint32_t kLeast = 17u * 1024u;      // the final sums of waves that share tiles
    a.ldsBytes = (off > kLeast ? off : kLeast) + 16u;
    a.dwTiles = tiles;
    a.partialFloats = tiles * 256u + groups * 16u + 16u;
    a.samples = samples;
    return a.ldsBytes <= 160u * 1024u;
}
inline bool planRound(const MlpArgs& m, int ct, RoundArgs& a, int& maxTiles)
{
    if (planRoundOf(kRoundSamples, m, ct, a, maxTiles)) return true;
    return ct == kF16 && m.numLayers >= 4 && planRoundOf(kRoundFewSamples, m, ct, a, maxTiles) && maxTiles > 4;
}

// Two workgroups to a compute unit where their LDS fits twice and a wave gets by with 128 registers.
constexpr int roundWavesPerSimd(int layers, int rt) { return rt == 2 && layers <= 3 ? 4 : 2; }
inline uint32_t roundWorkgroups(const RoundArgs& a, int layers, int rt, int numCUs)
{
    return (uint32_t)numCUs * (roundWavesPerSimd(layers, rt) == 4 && a.ldsBytes <= 80u * 1024u ? 2u : 1u);
}
inline int roundTiles(int maxTiles) { return maxTiles > 4 ? 4 : 2; }
// workgroups of a launch: no more than the batch has rounds
inline uint32_t roundBlocks(uint32_t batch, uint32_t samples, uint32_t resident)
{
    const uint32_t rounds = batch ? (batch - 1) / samples + 1 : 1;
    return rounds < resident ? rounds : resident;
}

template <typename T, int NL, int RT, int SAMPLES, bool ANY = false>
hipError_t launchRoundSized(hipStream_t stream, const TrainLaunch& t, RoundArgs& a, int numCUs)
{
    if constexpr (sizeof(T) == 2 && !ANY) {
        bool any = false;
        for (int l = 0; l < NL; ++l) any = any || (a.layers[l].shape.layout == kRowMajor && !roundWeightWhole<T>(a.layers[l]));
        if (any) return launchRoundSized<T, NL, RT, SAMPLES, true>(stream, t, a, numCUs);
    }
    constexpr int WAVES = roundWavesPerSimd(NL, RT);
    const hipError_t e = allowDynamicLds<trainRoundKernel<T, NL, RT, WAVES, SAMPLES, ANY>>(160 * 1024);
    if (e != hipSuccess) return e;
    const uint32_t blocks = roundBlocks(t.mlp.batch, SAMPLES, roundWorkgroups(a, NL, RT, numCUs));
    a.finish.numPartials = blocks;
    noteKernel(false, "trainRoundKernel<%s,%d layers,up to %d rows%s> + trainRoundReduceKernel",
               sizeof(T) == 4 ? "f32" : "f16", NL, 32 * RT, SAMPLES == kRoundFewSamples ? ",32 samples" : "");
    hipLaunchKernelGGL((trainRoundKernel<T, NL, RT, WAVES, SAMPLES, ANY>), dim3(blocks), dim3(kRoundThreads), a.ldsBytes, stream, a);
    const hipError_t e1 = hipGetLastError();
    if (e1 != hipSuccess) return e1;
    hipLaunchKernelGGL(trainRoundReduceKernel, dim3((a.partialFloats - 16u) / 64u + 1u), dim3(64 * kReduceWaves), 0, stream, a);
    return hipGetLastError();
}

// the arguments both kernels of a step read; false where planRound says so
template <typename T>
bool fillRoundArgs(const TrainLaunch& t, RoundArgs& a, int& maxTiles)
{
    if (!planRound(t.mlp, sizeof(T) == 4 ? kF32 : kF16, a, maxTiles)) return false;
    const int L = t.mlp.numLayers;
    a.in = t.mlp.in; a.inStride = t.mlp.inStride;
    a.targets = t.targets; a.targetStride = t.targetStride;
    a.batch = t.mlp.batch;
    const uint32_t rowBytes = (uint32_t)t.mlp.layers[0].in * (uint32_t)sizeof(T);
    a.inPieces = (rowBytes % 16u == 0u && t.mlp.inAlign >= 16u) ? (int32_t)(rowBytes / 16u) : 0;
    a.lossScale = t.lossScale;
    a.partials = t.workspace;
    a.wantLossMax = t.lossMax ? 1 : 0;
    for (int l = 0; l < L; ++l) a.finish.layers[l] = TrainReduceArgs::Layer{t.wGrad[l], t.bGrad[l], t.gradShape[l], t.mlp.layers[l].in, t.mlp.layers[l].out};
    a.finish.numLayers = L;
    a.finish.gradCt = t.gradCt;
    a.finish.partials = t.workspace;
    a.finish.lossSum = t.lossSum;
    a.finish.lossMax = t.lossMax;
    return true;
}

template <typename T>
hipError_t launchRoundTyped(hipStream_t stream, const TrainLaunch& t, int numCUs)
{
    constexpr int ct = sizeof(T) == 4 ? kF32 : kF16;
    RoundArgs a = {};
    int maxTiles = 0;
    if (!fillRoundArgs<T>(t, a, maxTiles)) return hipErrorInvalidValue;
    const int L = t.mlp.numLayers;
    if constexpr (sizeof(T) == 2) {
        if (a.samples == (uint32_t)kRoundFewSamples)
            return L == 4 ? launchRoundSized<T, 4, 4, kRoundFewSamples>(stream, t, a, numCUs) : launchRoundSized<T, 5, 4, kRoundFewSamples>(stream, t, a, numCUs);
    }
    switch (roundTiles(maxTiles) * 8 + L) {
#define CV_L(RT) case RT * 8 + 2: return launchRoundSized<T, 2, RT, kRoundSamples>(stream, t, a, numCUs); case RT * 8 + 3: return launchRoundSized<T, 3, RT, kRoundSamples>(stream, t, a, numCUs); \
                 case RT * 8 + 4: return launchRoundSized<T, 4, RT, kRoundSamples>(stream, t, a, numCUs); case RT * 8 + 5: return launchRoundSized<T, 5, RT, kRoundSamples>(stream, t, a, numCUs);
    CV_L(2) CV_L(4)
#undef CV_L
    }
    return hipErrorInvalidValue;
}

} // namespace
} // namespace cv
