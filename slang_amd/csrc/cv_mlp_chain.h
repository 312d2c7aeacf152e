// cv_mlp_chain.h -- fused forward MLP for any chain of FeedForwardLayer / FFLayer<T>
// (examples/mlp-training-coopvec/fflayer.slang:7-67, source/standard-modules/neural/layers.slang:34-110) of up to 128
// rows and columns without smooth activations, element type fp16, e4m3, fp32 or bfloat16.  Values and rounding points
// are those of mlpGenericKernel / mlpFloatKernel, bit for bit (same order of sums per accumulator).
//
// What bounds it: vector-ALU issue (conversion between layers; for T = float the split into F32Mma's pieces).  The run-time-size kernels
// spent most of their issue slots elsewhere: they computed tiles a layer does not have, formed an address and a mask for every input
// element of every tile, and waited for the inputs of a tile after asking for them.  Here
//   - a layer is a wave-uniform switch over its number of 16-row tiles MT; each arm is straight-line code for exactly
//     those tiles (k-tiles under one uniform branch each, which covers all accumulators and so copies none);
//   - inputs of whole, aligned groups of four (QUAD) come by buffer loads whose descriptor covers exactly the vectors of one 16-sample
//     tile: a lane's offsets are the same for every tile and are computed once, a slot beyond the vector has an offset outside the
//     descriptor and a sample beyond the batch lies outside it, and both read as zero without a compare or a mask;
//   - inputs of any other size come in reads of 16 (8) bytes at whatever element a lane's slots begin, which this chip takes at the
//     price of aligned ones, from a uniform address and one offset per lane; what lies behind the vector is masked off.  Reads that
//     would end behind the last vector are made ending there and shifted.  (One load per element before: 37-48-8 over 524 288 samples
//     fp16 32 -> 21 us, bf16 33 -> 22; masks on aligned inputs as well would cost 20-48-24-5 4 us of 49);
//   - matrices of 8 and 16 bits are staged with four chunks of a thread in flight, each one read where the matrix is RowMajor (cv_stage.h);
//   - results leave in pieces of four, two and one element, at whatever alignment they have;
//   - the loads of the next tiles are issued before the layers of the current ones;
//   - NT = 2 tiles share every weight fragment read from LDS and give the matrix pipeline twice the independent chains, for wide layers
//     and bfloat16 as well (T = float: one, for the registers of the pieces): 5-128-128-128-128-4 fp16 over 524 288 samples 148 -> 72 us,
//     with eight waves to a workgroup where one workgroup's weights fill a compute unit's LDS;
//   - leaky ReLU with a positive slope is a packed product and maximum (13-16-16-16-16-12 over 524 288 samples 30 -> 25 us).
// Measured against the run-time-size kernels: fp16 20-48-24-5 over 2 000 003 samples 78 -> 45 us; T = float, 20-48-24-5 over 2^20
// samples 91 us with v_mfma_f32_16x16x4_f32, 74 us with the pieces.  (Equal hidden layers: cv_mlp_equal_f32.h.)
// Networks of float whose pieces exceed the LDS (more than 52 fragments) split a fragment at every use, 52 vector instructions
// beside six matrix instructions, and are no faster than the fp32 instruction was: 64-128-128-64 over 2^18 samples 173 us (161),
// 128-128-128 183 (161), over 2^12 28.9 (20.1) and 29.5 us (20.3).  They stay on the pieces all the same, for the bits of the
// single-layer operators.
#pragma once
#include <type_traits>

#include "cv_matmul_impl.h"
#include "cv_mlp_generic_impl.h"

namespace cv {
namespace {

constexpr int kLeakyPacked = -1;                     // leaky ReLU with packedSlope(slope), beside the activations' own numbers
constexpr uint32_t kChainOutside = 0x80000000u;      // an offset no descriptor of a tile reaches

constexpr uint32_t kChainPieceDwords = (160 * 1024 - 512) / 4;      // a compute unit's LDS, less what the kernel declares itself

template <class Mma>
constexpr int chainComponent()
{
    return std::is_same<Mma, Bf16Mma>::value ? (int)kBF16 : (int)kF16;
}

// Four waves to a workgroup; up to eight for networks of float and of layers wider than 64, launched where the weights leave room for one
// workgroup in a compute unit's LDS, so that a SIMD still has two waves, one converting and splitting beside the other's matrix
// instructions (float, four waves / eight, 2^18 samples: 64-112-96-12 104 / 66 us, 96-80-72-16 106 / 63, split at use 64-128-128-64
// 282 / 173).
template <class Mma, int MAXT>
constexpr int chainThreads() { return Mma::kEsz == 4 || MAXT == 8 ? 512 : 256; }

template <int ACT>
__device__ __forceinline__ float chainActivateF32(float x, float slope)
{
    if constexpr (ACT == kActRelu) return F32Mma::relu(x);
    if constexpr (ACT == kActLeakyRelu) return fmaxf(x, x * slope);
    return x;
}

// four bfloat16 results: the activation of the rounded sums (ReLU commutes with the rounding)
template <int ACT>
__device__ __forceinline__ void bf16Results(const floatx4& z, float slope, uint32_t& p01, uint32_t& p23)
{
    if constexpr (ACT == kActLeakyRelu) {
        p01 = pack16<bf16_t>(activate16<bf16_t>(z[0], ACT, slope), activate16<bf16_t>(z[1], ACT, slope));
        p23 = pack16<bf16_t>(activate16<bf16_t>(z[2], ACT, slope), activate16<bf16_t>(z[3], ACT, slope));
    } else if constexpr (ACT == kActRelu) {
        p01 = pack16<bf16_t>(z[0] > 0.f ? z[0] : 0.f, z[1] > 0.f ? z[1] : 0.f);
        p23 = pack16<bf16_t>(z[2] > 0.f ? z[2] : 0.f, z[3] > 0.f ? z[3] : 0.f);
    } else {
        p01 = pack16<bf16_t>(z[0], z[1]);
        p23 = pack16<bf16_t>(z[2], z[3]);
    }
}

// One layer of float where some operand is beyond() (F32Careful); `act` holds pieces from decode<true>.
template <int MT, int KTS, bool PIECES>
__device__ __forceinline__ void carefulProduct(const uint32_t* wbase, const float* bbase, int KT, const uint32_t (&act)[KTS][F32Mma::kFD], floatx4 (&acc)[MT])
{
    constexpr int LANE_DW = PIECES ? F32Mma::kFD : F32Mma::kRawDW;
#pragma unroll 1
    for (int t = 0; t < MT; ++t) {
        const floatx4 bias = *(const floatx4*)(bbase + 16 * t);
        F32Careful c;
        c.start(bias);
#pragma unroll
        for (int kt = 0; kt < KTS; ++kt) {
            if (kt == 0 || kt < KT) c.template step<PIECES, true>(wbase + (size_t)(t * KT + kt) * 64 * LANE_DW, act[kt]);
        }
        const floatx4 r = c.finish(bias);
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[i] = t == i ? r : acc[i];
    }
}

// One layer of MT row tiles for NT sample tiles: `act` holds its B operands and receives the next layer's, or, for the
// last layer, the results are stored.
// PIECES (T = float): fragments lie in LDS as F32Mma's pieces; else as they lie in memory, split at every use.
// matBeyond, any (T = float): F32Mma::beyond of some layer's matrix, and of it or the vectors in `act`.
template <class Mma, int MAXT, int MT, int NT, bool PIECES>
__device__ __forceinline__ void chainLayer(const MlpArgs& a, const MlpLayerArgs& ly, const uint32_t* wbase, const float* bbase, int KT,
                                           bool last, int g, uint32_t sample, uint32_t (&act)[NT][MAXT / 2][Mma::kFD],
                                           bool matBeyond, bool& any)
{
    constexpr int FD = Mma::kFD, RAW = PIECES ? FD : Mma::kRawDW, MAXKT = MAXT / 2, OKT = (MT + 1) / 2;
    constexpr bool F32 = std::is_same<Mma, F32Mma>::value, BF16 = std::is_same<Mma, Bf16Mma>::value;
    floatx4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const floatx4 b = *(const floatx4*)(bbase + 16 * t);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[nt][t] = b;
    }
    if constexpr (F32) {
        // Fragments of G row tiles together and product by product, so that no matrix instruction waits for the one before it.
        static_assert(NT == 1, "one tile: two leave a SIMD fewer than two waves for their registers");
        constexpr int G = MT < 2 ? 1 : 2;
#pragma unroll
        for (int t0 = 0; t0 < MT; t0 += G) {
            F32Sum sum[G];
#pragma unroll
            for (int t = t0; t < MT && t < t0 + G; ++t) sum[t - t0] = SumOf<Mma>::start(acc[0][t]);
#pragma unroll
            for (int kt = 0; kt < MAXKT; ++kt) {
                if (kt == 0 || kt < KT) {
                    uint32_t w[G][FD];
#pragma unroll
                    for (int t = t0; t < MT && t < t0 + G; ++t) {
                        const uint32_t* raw = wbase + (size_t)(t * KT + kt) * 64 * RAW;
                        if constexpr (PIECES) {
#pragma unroll
                            for (int d = 0; d < FD; ++d) w[t - t0][d] = raw[d];
                        } else {
                            Mma::decode(raw, w[t - t0]);
                        }
                    }
                    staticFor<0, 6>([&](auto pc) {
#pragma unroll
                        for (int t = t0; t < MT && t < t0 + G; ++t) Mma::template product<decltype(pc)::value>(w[t - t0], act[0][kt], sum[t - t0]);
                    });
                }
            }
#pragma unroll
            for (int t = t0; t < MT && t < t0 + G; ++t) acc[0][t] = SumOf<Mma>::finish(sum[t - t0], acc[0][t]);
        }
        if (any) carefulProduct<MT, MAXKT, PIECES>(wbase, bbase, KT, act[0], acc[0]);      // (hardly ever: the rest stays straight-line code)
    } else
#pragma unroll
    for (int kt = 0; kt < MAXKT; ++kt) {
        if (kt == 0 || kt < KT) {
            // groups of row tiles whose fragments are read together, and no more registers than that takes
            constexpr int G = 4;
#pragma unroll
            for (int t0 = 0; t0 < MT; t0 += G) {
                uint32_t w[G][FD];
#pragma unroll
                for (int t = t0; t < MT && t < t0 + G; ++t) Mma::decode(wbase + (size_t)(t * KT + kt) * 64 * RAW, w[t - t0]);
#pragma unroll
                for (int t = t0; t < MT && t < t0 + G; ++t)
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) acc[nt][t] = Mma::mma(w[t - t0], act[nt][kt], acc[nt][t]);
            }
        }
    }

    // the activation is one of three, chosen once for all tiles
    auto finish = [&](auto actConst) {
        constexpr int ACT = decltype(actConst)::value;
        CarrierCfg cc{};
        if constexpr (!F32 && !BF16) {
            cc = makeCarrierCfg<Mma>(ly.act, ly.slope);
            cc.act = ACT;
            if (last) {            // the last layer's result is not re-quantised
                const half_t lo = ly.act == kActRelu ? (half_t)0.f : (half_t)-__builtin_inff();
                cc.floor2 = halfx2{lo, lo};
            }
        }
        if constexpr (F32) {
            if (!last) {
                float most = 0.f;
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int t = 0; t < MT; ++t) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[nt][t][r] = chainActivateF32<ACT>(acc[nt][t][r], ly.slope);
                        const u32x4 bits = __builtin_bit_cast(u32x4, acc[nt][t]);
                        const uint32_t raw[4] = {bits.x, bits.y, bits.z, bits.w};
                        most = Mma::largest(raw, 4, most);
                    }
                any = Mma::beyond(most);
                auto split = [&](auto anyConst) {
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                        for (int kt = 0; kt < OKT; ++kt) {
                            uint32_t raw[8];
#pragma unroll
                            for (int t = 0; t < 2; ++t) {    // (an odd number of tiles: the upper half of the last fragment is zero)
                                const u32x4 v = 2 * kt + t < MT ? __builtin_bit_cast(u32x4, acc[nt][2 * kt + t < MT ? 2 * kt + t : 0]) : u32x4{0u, 0u, 0u, 0u};
                                raw[4 * t] = v.x; raw[4 * t + 1] = v.y; raw[4 * t + 2] = v.z; raw[4 * t + 3] = v.w;
                            }
                            Mma::template decode<decltype(anyConst)::value>(raw, act[nt][kt]);
                        }
                };
                split(std::false_type());
                if (any) split(std::true_type());
                any = any | matBeyond;
                return;
            }
        }
        if (!last) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int kt = 0; kt < OKT; ++kt) {
                    const bool two = 2 * kt + 1 < MT;        // an odd number of tiles: the upper half of the last fragment is zero
                    const floatx4 x0 = acc[nt][2 * kt], x1 = two ? acc[nt][two ? 2 * kt + 1 : 2 * kt] : floatx4{0.f, 0.f, 0.f, 0.f};
                    if constexpr (BF16) {
                        bf16Results<ACT>(x0, ly.slope, act[nt][kt][0], act[nt][kt][1]);
                        if (two) bf16Results<ACT>(x1, ly.slope, act[nt][kt][2], act[nt][kt][3]);
                        else act[nt][kt][2] = act[nt][kt][3] = 0u;
                    } else {
                        halfx2 lo01, lo23, hi01 = {(half_t)0, (half_t)0}, hi23 = hi01;
                        carrierFromAcc<false, ACT == kLeakyPacked>(x0, cc, lo01, lo23);
                        if (two) carrierFromAcc<false, ACT == kLeakyPacked>(x1, cc, hi01, hi23);
                        if constexpr (!F32) fragFromCarrier<Mma>(lo01, lo23, hi01, hi23, cc, act[nt][kt]);
                    }
                }
            return;
        }
        const int row0 = g * 4 * MT;
        const bool quads = (ly.out & 3) == 0;      // (then a lane has four rows or none)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            const uint32_t s = sample + 16u * nt;
            if (s < a.batch) {
                uint8_t* o = a.out + (size_t)s * a.outStride + (size_t)row0 * (F32 ? 4 : 2);
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const int left = ly.out - row0 - 4 * t;      // rows of the result at and beyond this lane's four
                    if constexpr (F32) {
                        floatx4 z;
#pragma unroll
                        for (int r = 0; r < 4; ++r) z[r] = chainActivateF32<ACT>(acc[nt][t][r], ly.slope);
                        const u32x4 v = __builtin_bit_cast(u32x4, z);
                        uint8_t* const to = o + 16 * t;
                        if (left >= 4) {
                            ((Loose16<4>*)to)->v = v;
                        } else if (!quads && left > 0) {
                            if (left > 1) ((Loose8<4>*)to)->v = u32x2{v.x, v.y};
                            if (left != 2) ((uint32_t*)to)[left - 1] = left == 1 ? v.x : v.z;
                        }
                    } else {
                        uint32_t p[2];
                        if constexpr (BF16) {
                            bf16Results<ACT>(acc[nt][t], ly.slope, p[0], p[1]);
                        } else {
                            halfx2 p0, p1;
                            carrierFromAcc<false, ACT == kLeakyPacked>(acc[nt][t], cc, p0, p1);
                            p[0] = __builtin_bit_cast(uint32_t, p0);
                            p[1] = __builtin_bit_cast(uint32_t, p1);
                        }
                        uint8_t* const to = o + 8 * t;
                        if (left >= 4) {
                            ((Loose8<2>*)to)->v = u32x2{p[0], p[1]};
                        } else if (!quads && left > 0) {
                            if (left > 1) ((Loose4<2>*)to)->v = p[0];
                            if (left != 2) ((uint16_t*)to)[left - 1] = (uint16_t)(left == 1 ? p[0] : p[1]);
                        }
                    }
                }
            }
        }
    };
    if (!F32 && !BF16 && ly.act == kActLeakyRelu && packedSlope(ly.slope)) finish(std::integral_constant<int, kLeakyPacked>());
    else if (ly.act == kActLeakyRelu) finish(std::integral_constant<int, (int)kActLeakyRelu>());
    else if ((F32 || BF16) && ly.act == kActRelu) finish(std::integral_constant<int, (int)kActRelu>());
    else finish(std::integral_constant<int, (int)kActNone>());      // (half: ReLU is the floor of the carrier)
}

// MAXT: the bound on a layer's row tiles; NT: 16-sample tiles per wave and round.  INKT: the bound on the input's k-tiles.
// QUAD: input vectors of whole, aligned groups of four elements.
template <class Mma, int MAXT, int NT, bool PIECES, int INKT, bool QUAD>
__global__ __launch_bounds__((chainThreads<Mma, MAXT>()), Mma::kEsz == 4 ? (MAXT == 4 ? 3 : 2) : MAXT == 4 ? 4 : 2) void mlpChainKernel(const GenArgs ga)
{
    constexpr int MAXKT = MAXT / 2, FD = Mma::kFD, ESZ = Mma::kEsz, RAW = Mma::kRawDW;
    static_assert(Mma::kEpl == 8, "eight k-slots per lane and fragment");
    const MlpArgs& a = ga.mlp;
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    float* ldsB = (float*)(lds + ga.biasDwordBase);
    constexpr bool F32 = std::is_same<Mma, F32Mma>::value;
    constexpr int LANE_DW = PIECES ? FD : RAW;             // dwords per lane of a fragment in LDS
    const uint32_t threads = blockDim.x;
    const int L = a.numLayers;
    uint32_t most = 0u;
    if constexpr (F32) {
        for (int l = 0; l < L; ++l) {
            const MlpLayerArgs& ly = a.layers[l];
            const int MT = ga.gl[l].mt, KT = ga.gl[l].kt;
            uint32_t* const dst = lds + (size_t)ga.gl[l].fragBase * 64 * LANE_DW;
            if constexpr (PIECES) most = stageFragmentPieces(dst, ly.w, ly.shape, false, MT, KT, optGS((uint32_t)ly.in), (uint32_t)ly.out, (uint32_t)ly.in, 0, most);
            else stageFragments<ESZ, 8>(dst, ly.w, ly.shape, false, MT, KT, optGS((uint32_t)ly.in), (uint32_t)ly.out, (uint32_t)ly.in);
            for (int e = threadIdx.x; e < MT * 16; e += (int)threads) {
                const int row = ((e >> 2) & 3) * 4 * MT + 4 * (e >> 4) + (e & 3);
                ldsB[ga.gl[l].biasBase + e] = ly.bias && row < ly.out ? ((const float*)ly.bias)[row] : 0.f;
            }
        }
    } else {
        const int biases = ga.gl[L - 1].biasBase + ga.gl[L - 1].mt * 16;
        auto biasOf = [&](int e) {
            int l = 0;
            while (l + 1 < L && e >= (int)ga.gl[l + 1].biasBase) ++l;
            const MlpLayerArgs& ly = a.layers[l];
            const int at = e - (int)ga.gl[l].biasBase, MT = ga.gl[l].mt, row = ((at >> 2) & 3) * 4 * MT + 4 * (at >> 4) + (at & 3);
            return (ly.bias && row < ly.out) ? loadAsFloat(ly.bias + (size_t)row * 2, chainComponent<Mma>()) : 0.f;
        };
        const float firstBias = (int)threadIdx.x < biases ? biasOf(threadIdx.x) : 0.f;
        for (int l = 0; l < L; ++l) {
            const MlpLayerArgs& ly = a.layers[l];
            uint32_t* const dst = lds + (size_t)ga.gl[l].fragBase * 64 * LANE_DW;
            stageTogether<ESZ, 8>(ly.w, ly.shape, ga.gl[l].mt, ga.gl[l].kt, (uint32_t)ly.out, (uint32_t)ly.in,
                                  [&](int c, uint32_t (&v)[RAW]) { storeFragmentChunk<RAW>(dst + (size_t)c * RAW, v); });
        }
        if ((int)threadIdx.x < biases) ldsB[threadIdx.x] = firstBias;
        for (int e = threadIdx.x + (int)threads; e < biases; e += (int)threads) ldsB[e] = biasOf(e);
    }
    __syncthreads();
    bool matBeyond = false;
    if constexpr (F32) {
        if constexpr (!PIECES)
            for (uint32_t i = threadIdx.x; i < ga.biasDwordBase / RAW; i += threads) most = Mma::largestBits(lds + (size_t)i * RAW, RAW, most);
        matBeyond = __syncthreads_or(most >= Mma::kBeyondBits);
    }

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, n = lane & 15;
    const int in0 = a.layers[0].in, gs0 = (int)optGS((uint32_t)in0);
    // which of a lane's k-slots exist: in every lane all of the first wholeFragments fragments' ones
    const int colBase = g * gs0, validBytes = sliceBytes((uint32_t)in0, (uint32_t)gs0, (uint32_t)g, ESZ);
    const int wholeFragments = min(gs0, max(in0 - 3 * gs0, 0)) / 8;
    const uint64_t inEnd = vectorsEnd(a.batch, a.inStride, (uint32_t)in0, ESZ);
    const int kt0 = ga.gl[0].kt;
    const uint32_t laneOffset = (uint32_t)n * (uint32_t)a.inStride + (uint32_t)colBase * ESZ;
    // offsets of a lane's groups of four, the same for every tile (of float, where registers are scarce, formed for each)
    uint32_t off[QUAD && !F32 ? INKT : 1][2];
    if constexpr (QUAD && !F32) {
#pragma unroll
        for (int kt = 0; kt < INKT; ++kt)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int q = (kt * 8 + u * 4) * ESZ;
                off[kt][u] = q < validBytes ? laneOffset + q : kChainOutside;
            }
    }
    // (8 and 16 bits: the bytes of a lane's fragments that exist, where there are registers for them)
    constexpr int MASKS = QUAD || F32 || (ESZ == 2 && NT == 2 && INKT > 1) ? 0 : INKT;
    uint32_t mask[MASKS > 0 ? MASKS : 1][RAW];
#pragma unroll
    for (int kt = 0; kt < MASKS; ++kt) {
#pragma unroll
        for (int d = 0; d < RAW; ++d) mask[kt][d] = 0xffffffffu;
        clearBehind<ESZ>(mask[kt], validBytes - kt * 8 * ESZ);
    }

    const uint32_t numTiles = (uint32_t)(((uint64_t)a.batch + 15) / 16), waves = threads / 64u, step = gridDim.x * waves * NT;
    uint32_t raw[NT][INKT][RAW] = {};
    const bool halfTail = gs0 - 8 * (kt0 - 1) <= 4;
    auto fetch = [&](uint32_t tile) {
        uint32_t lane0 = laneOffset;
        if constexpr (F32) asm volatile("" : "+v"(lane0));      // (else the compiler keeps every address over the tiles)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            if constexpr (QUAD) {
                const uint32_t first = min(tile + nt, numTiles - 1) * 16u;
                const uint32_t rows = tile + nt < numTiles ? min(16u, a.batch - first) : 0u;
                const uint32_t bytes = rows ? (rows - 1) * (uint32_t)a.inStride + (uint32_t)in0 * ESZ : 0u;
                const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc((void*)(a.in + (size_t)first * a.inStride), 0, bytes, 0x00027000);
#pragma unroll
                for (int kt = 0; kt < INKT; ++kt)
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        if (kt > 0 && kt >= kt0) continue;       // (wave-uniform; empty loads of absent k-tiles cost 6 us of 51)
                        uint32_t* r = raw[nt][kt] + u * (RAW / 2);
                        if constexpr (F32) {
                            const int q = (kt * 8 + u * 4) * ESZ;
                            const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(src, q < validBytes ? lane0 + q : kChainOutside, 0, 0));
                            r[0] = v.x; r[1] = v.y; r[2] = v.z; r[3] = v.w;
                        } else if constexpr (ESZ == 2) {
                            const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(src, off[kt][u], 0, 0));
                            r[0] = v.x; r[1] = v.y;
                        } else {
                            r[0] = __builtin_amdgcn_raw_buffer_load_b32(src, off[kt][u], 0, 0);
                        }
                    }
                continue;
            }
            const uint32_t first = min(tile + nt, numTiles - 1) * 16u;      // (beyond the batch: the last tile, whose results nobody stores)
            // reads of 16 bytes (8) at whatever element a lane's slots begin; what would end behind the last vector is read ending there and moved down (loadUpTo)
            if (tileReadsEnd(first, 16u, a.inStride, (uint32_t)gs0, (uint32_t)(8 * kt0), ESZ) <= inEnd) {
                const uint8_t* base = a.in + (uint64_t)first * a.inStride;
#pragma unroll
                for (int kt = 0; kt < INKT; ++kt) {
                    if (kt > 0 && kt >= kt0) continue;       // (wave-uniform)
                    const uint8_t* q = base + lane0 + kt * 8 * ESZ;
                    if (kt + 1 == kt0 && halfTail) {      // (no lane has slots in the upper half of the last fragment)
                        if constexpr (ESZ == 4) { const u32x4 v = ((const Loose16<ESZ>*)q)->v; raw[nt][kt][0] = v.x; raw[nt][kt][1] = v.y; raw[nt][kt][2] = v.z; raw[nt][kt][3] = v.w; }
                        else if constexpr (ESZ == 2) { const u32x2 v = ((const Loose8<ESZ>*)q)->v; raw[nt][kt][0] = v.x; raw[nt][kt][1] = v.y; }
                        else raw[nt][kt][0] = ((const Loose4<ESZ>*)q)->v;
                    } else {
                        loadLoose<ESZ>(q, raw[nt][kt]);
                    }
                }
            } else {
                const uint8_t* q = a.in + (uint64_t)min(first + n, a.batch - 1u) * a.inStride + colBase * ESZ;
#pragma unroll
                for (int kt = 0; kt < INKT; ++kt) {
                    if (kt > 0 && kt >= kt0) continue;
                    if (inEnd >= 16u) loadUpTo<ESZ>(q + kt * 8 * ESZ, a.in + inEnd, raw[nt][kt]);
                    else loadSlots<RAW>(raw[nt][kt], q + kt * 8 * ESZ, validBytes - kt * 8 * ESZ, 2);
                }
            }
        }
    };

    uint32_t tile = (blockIdx.x * waves + wave) * NT;
    if (tile >= numTiles) return;
    // (not ahead for more than 64 inputs of float: the registers would be spilled ones, and the other wave's work covers the wait)
    constexpr bool AHEAD = !F32 || INKT <= 2;
    if constexpr (AHEAD) fetch(tile);
    for (;;) {
        if constexpr (!AHEAD) fetch(tile);
        uint32_t act[NT][MAXKT][FD];
        bool any = matBeyond;
        if constexpr (!QUAD) {
            int valid = validBytes;
            if constexpr (MASKS < INKT) pinHere(valid);      // (comparisons with it stay in the loop: hoisted, they take more scalar registers than there are)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int kt = 0; kt < INKT; ++kt)
                    if ((kt == 0 || kt < kt0) && kt >= wholeFragments) {
                        if (kt < MASKS) {
#pragma unroll
                            for (int d = 0; d < RAW; ++d) raw[nt][kt][d] &= mask[kt < MASKS ? kt : 0][d];
                        } else {
                            clearBehind<ESZ>(raw[nt][kt], valid - kt * 8 * ESZ);
                        }
                    }
        }
        if constexpr (F32) {
            float most = 0.f;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int kt = 0; kt < INKT; ++kt)
                    if (kt == 0 || kt < kt0) most = Mma::largest(raw[nt][kt], RAW, most);
            any = any | Mma::beyond(most);
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int kt = 0; kt < INKT; ++kt) {
                if (F32 && kt > 0 && kt >= kt0) continue;
                Mma::decode(raw[nt][kt], act[nt][kt]);
                if constexpr (F32) {
                    if (any) Mma::template decode<true>(raw[nt][kt], act[nt][kt]);
                }
            }
        const uint64_t following = (uint64_t)tile + step;
        const uint32_t next = following < numTiles ? (uint32_t)following : numTiles;
        if constexpr (AHEAD) fetch(next);                     // (beyond the batch: QUAD's descriptor is empty and nothing is read; else the last tile again)

        const uint32_t sample = tile * 16u + n;
        for (int l = 0; l < L; ++l) {
            const MlpLayerArgs& ly = a.layers[l];
            const uint32_t* wbase = lds + ((size_t)ga.gl[l].fragBase * 64 + lane) * LANE_DW;
            const float* bbase = ldsB + ga.gl[l].biasBase + 4 * g;
            const int KT = ga.gl[l].kt;
            const bool last = l + 1 == L;
#define CV_CHAIN_ARM(mt_) case mt_: chainLayer<Mma, MAXT, mt_, NT, PIECES>(a, ly, wbase, bbase, KT, last, g, sample, act, matBeyond, any); break;
            if constexpr (MAXT == 4) {
                switch (ga.gl[l].mt) { CV_CHAIN_ARM(1) CV_CHAIN_ARM(2) CV_CHAIN_ARM(3) CV_CHAIN_ARM(4) }
            } else {
                switch (ga.gl[l].mt) {
                    CV_CHAIN_ARM(1) CV_CHAIN_ARM(2) CV_CHAIN_ARM(3) CV_CHAIN_ARM(4)
                    CV_CHAIN_ARM(5) CV_CHAIN_ARM(6) CV_CHAIN_ARM(7) CV_CHAIN_ARM(8)
                }
            }
#undef CV_CHAIN_ARM
        }
        if (next >= numTiles) break;
        tile = next;
    }
}

template <class Mma, int MAXT, int NT, bool PIECES, int INKT, bool QUAD>
hipError_t launchChainSized(hipStream_t stream, const GenArgs& ga, size_t ldsBytes, int numCUs)
{
    const hipError_t ea = allowDynamicLds<mlpChainKernel<Mma, MAXT, NT, PIECES, INKT, QUAD>>((int)((PIECES ? kChainPieceDwords : kGenLdsDwords) * 4));
    if (ea != hipSuccess) return ea;
    const uint32_t numTiles = (uint32_t)(((uint64_t)ga.mlp.batch + 15) / 16);
    const uint32_t waves = chainThreads<Mma, MAXT>() == 512 && ldsBytes > 80 * 1024 ? 8u : 4u;
    int perCU = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, mlpChainKernel<Mma, MAXT, NT, PIECES, INKT, QUAD>, (int)(64 * waves), ldsBytes) != hipSuccess || perCU < 1) perCU = 1;
    const uint32_t need = (numTiles + waves * NT - 1) / (waves * NT), cap = (uint32_t)numCUs * (uint32_t)perCU;
    noteKernel(false, "mlpChainKernel<%s,up to %d rows,NT=%d%s>", Mma::kName, 16 * MAXT, NT, PIECES || Mma::kEsz < 4 ? "" : ",split at use");
    hipLaunchKernelGGL((mlpChainKernel<Mma, MAXT, NT, PIECES, INKT, QUAD>), dim3(need < cap ? need : cap), dim3(64 * waves), ldsBytes, stream, ga);
    return hipGetLastError();
}

template <class Mma, int MAXT, bool PIECES>
hipError_t launchChainRows(hipStream_t stream, const GenArgs& ga, size_t ldsBytes, int numCUs)
{
    constexpr uint32_t ESZ = Mma::kEsz;
    // Two tiles per wave as soon as every SIMD has two waves of them; below that the tiles are spread over the chip.
    // (One for fp32, where two would leave a SIMD one wave for their registers)
    auto sized = [&](auto quadConst) {
        constexpr bool QUAD = decltype(quadConst)::value;
        constexpr int ALL = MAXT / 2;
        const int kt0 = ga.gl[0].kt;
        if constexpr (ESZ < 4) {
            // (up to 32 inputs: fewer registers for the vectors on their way)
            if ((uint64_t)ga.mlp.batch > (uint64_t)numCUs * 8 * 16)
                return kt0 == 1 ? launchChainSized<Mma, MAXT, 2, PIECES, 1, QUAD>(stream, ga, ldsBytes, numCUs) : launchChainSized<Mma, MAXT, 2, PIECES, ALL, QUAD>(stream, ga, ldsBytes, numCUs);
            if (kt0 == 1) return launchChainSized<Mma, MAXT, 1, PIECES, 1, QUAD>(stream, ga, ldsBytes, numCUs);
        } else if constexpr (MAXT == 8) {
            // (up to 64 inputs before wide layers of float: the registers of the other k-tiles would be spilled ones)
            if (kt0 <= 2) return launchChainSized<Mma, MAXT, 1, PIECES, 2, QUAD>(stream, ga, ldsBytes, numCUs);
        }
        return launchChainSized<Mma, MAXT, 1, PIECES, ALL, QUAD>(stream, ga, ldsBytes, numCUs);
    };
    return ga.mlp.layers[0].in % 4 == 0 && ga.mlp.inAlign >= 4 * ESZ ? sized(std::true_type()) : sized(std::false_type());
}

// hipErrorInvalidValue for calls this kernel does not take: smooth activations, inputs that are encoded or quantised on
// the way, layers beyond 128, networks beyond 144 KB of LDS, strides above 2^26 bytes
template <class Mma>
hipError_t launchChain(hipStream_t stream, const MlpArgs& a, int numCUs)
{
    if (hasSmoothActivation(a) || a.inEncoding != kEncodeNone || a.inHalfAsE4M3 || a.inStride > (1u << 26)) return hipErrorInvalidValue;
    GenArgs ga{};
    uint32_t widest = 0;
    // (the pieces of a network of float take half as much again: where they do not fit, fragments stay as they are in memory)
    if constexpr (Mma::kEsz == 4) {
        const uint32_t dwords = planGeneric<Mma>(a, ga, kChainPieceDwords, &widest, Mma::kFD);
        if (dwords)
            return widest <= 4 ? launchChainRows<Mma, 4, true>(stream, ga, (size_t)dwords * 4, numCUs) : launchChainRows<Mma, 8, true>(stream, ga, (size_t)dwords * 4, numCUs);
    }
    const uint32_t dwords = planGeneric<Mma>(a, ga, kGenLdsDwords, &widest);
    if (!dwords) return hipErrorInvalidValue;
    return widest <= 4 ? launchChainRows<Mma, 4, false>(stream, ga, (size_t)dwords * 4, numCUs) : launchChainRows<Mma, 8, false>(stream, ga, (size_t)dwords * 4, numCUs);
}

} // namespace
} // namespace cv
