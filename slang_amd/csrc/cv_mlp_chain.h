// cv_mlp_chain.h -- fused forward MLP for any chain of FeedForwardLayer / FFLayer<T>
// (examples/mlp-training-coopvec/fflayer.slang:7-67, source/standard-modules/neural/layers.slang:34-110) of up to 128
// rows and columns without smooth activations, element type fp16, e4m3, fp32 or bfloat16.  Values and rounding points
// are those of mlpGenericKernel / mlpFloatKernel, bit for bit (same order of sums per accumulator).
//
// What bounds it: vector-ALU issue for 16- and 8-bit elements (conversion between layers), the fp32 matrix
// instructions for T = float.  The run-time-size kernels spent most of their issue slots elsewhere: they computed tiles
// a layer does not have, formed an address and a mask for every input element of every tile, and waited for the inputs
// of a tile after asking for them.  Here
//   - a layer is a wave-uniform switch over its number of 16-row tiles MT; each arm is straight-line code for exactly
//     those tiles (k-tiles under one uniform branch each, which covers all accumulators and so copies none);
//   - input loads are buffer loads whose descriptor covers exactly the vectors of one 16-sample tile: a lane's offsets
//     are the same for every tile and are computed once, a slot beyond the vector has an offset outside the
//     descriptor and a sample beyond the batch lies outside it, and both read as zero without a compare or a mask;
//   - the loads of the next tiles are issued before the layers of the current ones;
//   - NT = 2 tiles share every weight fragment read from LDS and give the matrix pipeline twice the independent chains.
// Measured against the run-time-size kernels: fp32 32-64-64-8 over 2^22 samples 729 -> 522 us (115 TFLOP/s of padded
// layers, 73 % of what v_mfma_f32_16x16x4_f32 issues at most), fp16 20-48-24-5 over 2 000 003 samples 78 -> 45 us.
#pragma once
#include <type_traits>

#include "cv_matmul_impl.h"
#include "cv_mlp_generic_impl.h"

namespace cv {
namespace {

constexpr uint32_t kChainOutside = 0x80000000u;      // an offset no descriptor of a tile reaches

template <class Mma>
constexpr int chainComponent()
{
    return std::is_same<Mma, F32Mma>::value ? (int)kF32 : std::is_same<Mma, Bf16Mma>::value ? (int)kBF16 : (int)kF16;
}

template <int ACT>
__device__ __forceinline__ float chainActivateF32(float x, float slope)
{
    if constexpr (ACT == kActRelu) return x > 0.f ? x : 0.f;
    if constexpr (ACT == kActLeakyRelu) return fmaxf(x, x * slope);
    return x;
}

// One layer of MT row tiles for NT sample tiles: `act` holds its B operands and receives the next layer's, or, for the
// last layer, the results are stored.
template <class Mma, int MAXT, int MT, int NT>
__device__ __forceinline__ void chainLayer(const MlpArgs& a, const MlpLayerArgs& ly, const uint32_t* wbase, const float* bbase, int KT,
                                           bool last, bool quads, int g, uint32_t sample, uint32_t (&act)[NT][MAXT / 2][Mma::kFD])
{
    constexpr int FD = Mma::kFD, RAW = Mma::kRawDW, MAXKT = MAXT / 2, OKT = (MT + 1) / 2;
    constexpr bool F32 = std::is_same<Mma, F32Mma>::value, BF16 = std::is_same<Mma, Bf16Mma>::value;
    floatx4 acc[NT][MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const floatx4 b = *(const floatx4*)(bbase + 16 * t);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[nt][t] = b;
    }
#pragma unroll
    for (int kt = 0; kt < MAXKT; ++kt) {
        if (kt == 0 || kt < KT) {
            // groups of row tiles whose fragments are read together: four sums side by side, so that none of fp32's eight
            // matrix instructions per fragment waits for the one before it, and no more registers than that takes
            constexpr int G = F32 && NT == 2 ? 2 : 4;
#pragma unroll
            for (int t0 = 0; t0 < MT; t0 += G) {
                uint32_t w[G][FD];
#pragma unroll
                for (int t = t0; t < MT && t < t0 + G; ++t) Mma::decode(wbase + (size_t)(t * KT + kt) * 64 * RAW, w[t - t0]);
                if constexpr (F32) {
#pragma unroll
                    for (int s = 0; s < 8; ++s)
#pragma unroll
                        for (int t = t0; t < MT && t < t0 + G; ++t)
#pragma unroll
                            for (int nt = 0; nt < NT; ++nt)
                                acc[nt][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, w[t - t0][s]),
                                                                                  __builtin_bit_cast(float, act[nt][kt][s]), acc[nt][t], 0, 0, 0);
                } else {
#pragma unroll
                    for (int t = t0; t < MT && t < t0 + G; ++t)
#pragma unroll
                        for (int nt = 0; nt < NT; ++nt) acc[nt][t] = Mma::mma(w[t - t0], act[nt][kt], acc[nt][t]);
                }
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
        if (!last) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int kt = 0; kt < OKT; ++kt) {
                    const bool two = 2 * kt + 1 < MT;        // an odd number of tiles: the upper half of the last fragment is zero
                    const floatx4 x0 = acc[nt][2 * kt], x1 = two ? acc[nt][two ? 2 * kt + 1 : 2 * kt] : floatx4{0.f, 0.f, 0.f, 0.f};
                    if constexpr (F32) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            act[nt][kt][r] = __builtin_bit_cast(uint32_t, chainActivateF32<ACT>(x0[r], ly.slope));
                            act[nt][kt][4 + r] = two ? __builtin_bit_cast(uint32_t, chainActivateF32<ACT>(x1[r], ly.slope)) : 0u;
                        }
                    } else if constexpr (BF16) {
                        float z[8];
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            z[r] = activate16<bf16_t>(x0[r], ACT, ly.slope);
                            z[4 + r] = two ? activate16<bf16_t>(x1[r], ACT, ly.slope) : 0.f;
                        }
#pragma unroll
                        for (int d = 0; d < 4; ++d) act[nt][kt][d] = pack16<bf16_t>(z[2 * d], z[2 * d + 1]);
                    } else {
                        halfx2 lo01, lo23, hi01 = {(half_t)0, (half_t)0}, hi23 = hi01;
                        carrierFromAcc<false>(x0, cc, lo01, lo23);
                        if (two) carrierFromAcc<false>(x1, cc, hi01, hi23);
                        fragFromCarrier<Mma>(lo01, lo23, hi01, hi23, cc, act[nt][kt]);
                    }
                }
            return;
        }
        const int row0 = g * 4 * MT;
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
                        if (quads) {
                            if (left > 0) *(floatx4*)(o + 16 * t) = z;
                        } else {
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                if (r < left) ((float*)o)[4 * t + r] = z[r];
                        }
                    } else {
                        uint32_t p[2];
                        if constexpr (BF16) {
                            p[0] = pack16<bf16_t>(activate16<bf16_t>(acc[nt][t][0], ACT, ly.slope), activate16<bf16_t>(acc[nt][t][1], ACT, ly.slope));
                            p[1] = pack16<bf16_t>(activate16<bf16_t>(acc[nt][t][2], ACT, ly.slope), activate16<bf16_t>(acc[nt][t][3], ACT, ly.slope));
                        } else {
                            halfx2 p0, p1;
                            carrierFromAcc<false>(acc[nt][t], cc, p0, p1);
                            p[0] = __builtin_bit_cast(uint32_t, p0);
                            p[1] = __builtin_bit_cast(uint32_t, p1);
                        }
                        if (quads) {
                            if (left > 0) *(u32x2*)(o + 8 * t) = u32x2{p[0], p[1]};
                        } else {
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                if (r < left) ((uint16_t*)o)[4 * t + r] = (uint16_t)(p[r / 2] >> (16 * (r & 1)));
                        }
                    }
                }
            }
        }
    };
    if (ly.act == kActLeakyRelu) finish(std::integral_constant<int, (int)kActLeakyRelu>());
    else if ((F32 || BF16) && ly.act == kActRelu) finish(std::integral_constant<int, (int)kActRelu>());
    else finish(std::integral_constant<int, (int)kActNone>());      // (half: ReLU is the floor of the carrier)
}

// MAXT: the bound on a layer's row tiles; NT: 16-sample tiles per wave and round; QUAD: input vectors of whole, aligned
// groups of four elements, which one load takes (else one load per element, any size and alignment).
// fp32 up to 64 wide: three waves per SIMD, four registers short of it, measure 522 us where two without a spill take 554.
template <class Mma, int MAXT, int NT, bool QUAD>
__global__ __launch_bounds__(256, (Mma::kEsz == 4 && MAXT == 4 && QUAD) ? 3 : 1) void mlpChainKernel(const GenArgs ga)
{
    constexpr int MAXKT = MAXT / 2, FD = Mma::kFD, ESZ = Mma::kEsz, RAW = Mma::kRawDW;
    constexpr int UNITS = QUAD ? 2 : 8;                    // loads per fragment
    constexpr int UDW = QUAD ? RAW / 2 : 1;                // dwords of registers a load fills
    static_assert(Mma::kEpl == 8, "eight k-slots per lane and fragment");
    const MlpArgs& a = ga.mlp;
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    float* ldsB = (float*)(lds + ga.biasDwordBase);
    for (int l = 0; l < a.numLayers; ++l) {
        const MlpLayerArgs& ly = a.layers[l];
        const int MT = ga.gl[l].mt, KT = ga.gl[l].kt;
        stageFragments<ESZ, 8>(lds + ga.gl[l].fragBase * 64 * RAW, ly.w, ly.shape, false, MT, KT, optGS((uint32_t)ly.in),
                               (uint32_t)ly.out, (uint32_t)ly.in);
        for (int e = threadIdx.x; e < MT * 16; e += 256) {
            const int t = e >> 4, gg = (e >> 2) & 3, r = e & 3, row = gg * 4 * MT + 4 * t + r;
            ldsB[ga.gl[l].biasBase + e] = (ly.bias && row < ly.out) ? loadAsFloat(ly.bias + (size_t)row * (chainComponent<Mma>() == kF32 ? 4 : 2), chainComponent<Mma>()) : 0.f;
        }
    }
    __syncthreads();

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, n = lane & 15;
    const int L = a.numLayers;
    const uint32_t in0 = (uint32_t)a.layers[0].in, gs0 = optGS(in0), rowBytes = in0 * ESZ;
    const bool quads = a.layers[L - 1].out % 4 == 0 && a.outAlign >= (std::is_same<Mma, F32Mma>::value ? 16u : 8u);

    uint32_t off[MAXKT][UNITS];
#pragma unroll
    for (int kt = 0; kt < MAXKT; ++kt)
#pragma unroll
        for (int u = 0; u < UNITS; ++u) {
            const uint32_t q = kt * 8 + u * (8 / UNITS), col = g * gs0 + q;
            off[kt][u] = q < gs0 && col < in0 ? (uint32_t)n * (uint32_t)a.inStride + col * ESZ : kChainOutside;
        }

    const uint32_t numTiles = (uint32_t)(((uint64_t)a.batch + 15) / 16), step = gridDim.x * 4u * NT;
    const int kt0 = ga.gl[0].kt;
    uint32_t raw[NT][MAXKT][UNITS * UDW];
    auto fetch = [&](uint32_t tile) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            // the vectors of this tile that exist: none for a tile beyond the batch
            const uint32_t first = min(tile + nt, numTiles - 1) * 16u;
            const uint32_t rows = tile + nt < numTiles ? min(16u, a.batch - first) : 0u;
            const uint32_t bytes = rows ? (rows - 1) * (uint32_t)a.inStride + rowBytes : 0u;
            const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc((void*)(a.in + (size_t)first * a.inStride), 0, bytes, 0x00027000);
#pragma unroll
            for (int kt = 0; kt < MAXKT; ++kt)
#pragma unroll
                for (int u = 0; u < UNITS; ++u) {
                    if (kt > 0 && kt >= kt0) continue;       // (wave-uniform; empty loads of absent k-tiles cost 6 us of 51)
                    uint32_t* r = raw[nt][kt] + u * UDW;
                    if constexpr (QUAD && ESZ == 4) {
                        const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(src, off[kt][u], 0, 0));
                        r[0] = v.x; r[1] = v.y; r[2] = v.z; r[3] = v.w;
                    } else if constexpr (QUAD && ESZ == 2) {
                        const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(src, off[kt][u], 0, 0));
                        r[0] = v.x; r[1] = v.y;
                    } else if constexpr (QUAD || ESZ == 4) {
                        r[0] = __builtin_amdgcn_raw_buffer_load_b32(src, off[kt][u], 0, 0);
                    } else if constexpr (ESZ == 2) {
                        r[0] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(src, off[kt][u], 0, 0);
                    } else {
                        r[0] = (uint8_t)__builtin_amdgcn_raw_buffer_load_b8(src, off[kt][u], 0, 0);
                    }
                }
        }
    };

    uint32_t tile = (blockIdx.x * 4u + wave) * NT;
    if (tile >= numTiles) return;
    fetch(tile);
    for (;;) {
        uint32_t act[NT][MAXKT][FD];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int kt = 0; kt < MAXKT; ++kt) {
                if constexpr (QUAD || ESZ == 4) {
                    Mma::decode(raw[nt][kt], act[nt][kt]);
                } else {
                    uint32_t packed[RAW];
#pragma unroll
                    for (int d = 0; d < RAW; ++d) {
                        const uint32_t* r = raw[nt][kt] + d * (4 / ESZ);
                        if constexpr (ESZ == 2) packed[d] = r[0] | r[1] << 16;
                        else packed[d] = r[0] | r[1] << 8 | r[2] << 16 | r[3] << 24;
                    }
                    Mma::decode(packed, act[nt][kt]);
                }
            }
        const uint64_t following = (uint64_t)tile + step;
        const uint32_t next = following < numTiles ? (uint32_t)following : numTiles;
        fetch(next);                     // (beyond the batch: an empty descriptor, nothing is read)

        const uint32_t sample = tile * 16u + n;
        for (int l = 0; l < L; ++l) {
            const MlpLayerArgs& ly = a.layers[l];
            const uint32_t* wbase = lds + ((size_t)ga.gl[l].fragBase * 64 + lane) * RAW;
            const float* bbase = ldsB + ga.gl[l].biasBase + 4 * g;
            const int KT = ga.gl[l].kt;
            const bool last = l + 1 == L;
#define CV_CHAIN_ARM(mt_) case mt_: chainLayer<Mma, MAXT, mt_, NT>(a, ly, wbase, bbase, KT, last, quads, g, sample, act); break;
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

template <class Mma, int MAXT, int NT, bool QUAD>
hipError_t launchChainSized(hipStream_t stream, const GenArgs& ga, size_t ldsBytes, int numCUs)
{
    const hipError_t ea = allowDynamicLds<mlpChainKernel<Mma, MAXT, NT, QUAD>>((int)(kGenLdsDwords * 4));
    if (ea != hipSuccess) return ea;
    int perCU = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, mlpChainKernel<Mma, MAXT, NT, QUAD>, 256, ldsBytes) != hipSuccess || perCU < 1) perCU = 1;
    const uint32_t numTiles = (uint32_t)(((uint64_t)ga.mlp.batch + 15) / 16), need = (numTiles + 4 * NT - 1) / (4 * NT);
    const uint32_t cap = (uint32_t)numCUs * (uint32_t)perCU;
    noteKernel(false, "mlpChainKernel<%s,up to %d rows,NT=%d%s>", Mma::kName, 16 * MAXT, NT,
               QUAD ? ",loads of four elements" : "");
    hipLaunchKernelGGL((mlpChainKernel<Mma, MAXT, NT, QUAD>), dim3(need < cap ? need : cap), dim3(256), ldsBytes, stream, ga);
    return hipGetLastError();
}

template <class Mma, int MAXT>
hipError_t launchChainRows(hipStream_t stream, const GenArgs& ga, size_t ldsBytes, int numCUs)
{
    constexpr uint32_t ESZ = Mma::kEsz;
    const MlpArgs& a = ga.mlp;
    const bool quad = a.layers[0].in % 4 == 0 && a.inAlign >= 4 * ESZ;
    // Two tiles per wave as soon as every SIMD has two waves of them; below that the tiles are spread over the chip.
    // (One where two would leave a SIMD one wave for their registers: fp32 layers wider than 64, and layers wider than 64
    // whose input comes element by element)
    if ((uint64_t)a.batch > (uint64_t)numCUs * 8 * 16) {
        if constexpr (MAXT == 4) {
            if (!quad) return launchChainSized<Mma, MAXT, 2, false>(stream, ga, ldsBytes, numCUs);
        }
        if constexpr (MAXT == 4 || ESZ < 4) {
            if (quad) return launchChainSized<Mma, MAXT, 2, true>(stream, ga, ldsBytes, numCUs);
        }
    }
    return quad ? launchChainSized<Mma, MAXT, 1, true>(stream, ga, ldsBytes, numCUs) : launchChainSized<Mma, MAXT, 1, false>(stream, ga, ldsBytes, numCUs);
}

// hipErrorInvalidValue for calls this kernel does not take: smooth activations, inputs that are encoded or quantised on
// the way, layers beyond 128, networks beyond 144 KB of LDS, strides whose 16 vectors an offset of 31 bits does not span
template <class Mma>
hipError_t launchChain(hipStream_t stream, const MlpArgs& a, int numCUs)
{
    if (hasSmoothActivation(a) || a.inEncoding != kEncodeNone || a.inHalfAsE4M3 || a.inStride > (1u << 26)) return hipErrorInvalidValue;
    GenArgs ga{};
    uint32_t widest = 0;
    const uint32_t dwords = planGeneric<Mma>(a, ga, kGenLdsDwords, &widest);
    if (!dwords) return hipErrorInvalidValue;
    return widest <= 4 ? launchChainRows<Mma, 4>(stream, ga, (size_t)dwords * 4, numCUs) : launchChainRows<Mma, 8>(stream, ga, (size_t)dwords * 4, numCUs);
}

} // namespace
} // namespace cv
