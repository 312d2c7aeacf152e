// cv_mlp_equal_f32.h -- fused forward network of float whose hidden layers are equally many 16-row tiles: the shape of most
// networks (8-64-64-64-3, 32-64-64-8, ...), in front of mlpChainKernel (cv_mlp_chain.h), which takes any.  Same bits.
//
// What bounds it: vector-ALU issue.  Between two layers every value is activated and split into three bfloat16 pieces
// (F32Mma: 5.5 instructions a value), and the matrix instructions, six for 16 rows, 16 samples and 32 terms, issue through the
// same port.  The any-shape kernel spends a third as much again on copying registers: every number of row tiles is another
// arm of a switch, whose results meet behind it.  Here the hidden layers are one straight-line body, run once per layer, 16
// samples to a wave and four waves per SIMD (128 registers), so that one wave's matrix instructions run beside
// another's conversions.  32-64-64-8 over 2^22 samples: 523 us on v_mfma_f32_16x16x4_f32 in the any-shape kernel, 402 us there with the
// pieces, 367 us here; 8-64-64-64-64-3 over 2^20: 276, 276, 161 us.
#pragma once
#include "cv_mlp_chain.h"

namespace cv {
namespace {

// One layer of KT k-tiles and MT row tiles: acc = W act + bias.  Two row tiles together, product by product.
template <int KT, int MT>
__device__ __forceinline__ void equalProduct(const uint32_t* wbase, const float* bbase, const uint32_t (&act)[KT][F32Mma::kFD], bool any, floatx4 (&acc)[MT])
{
    constexpr int FD = F32Mma::kFD, G = MT < 2 ? 1 : 2;
#pragma unroll
    for (int t0 = 0; t0 < MT; t0 += G) {
        F32Sum sum[G];
#pragma unroll
        for (int t = t0; t < t0 + G; ++t) sum[t - t0] = SumOf<F32Mma>::start(floatx4{});
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
            uint32_t w[G][FD];
#pragma unroll
            for (int t = t0; t < t0 + G; ++t)
#pragma unroll
                for (int d = 0; d < FD; ++d) w[t - t0][d] = wbase[(size_t)(t * KT + kt) * 64 * FD + d];
            staticFor<0, 6>([&](auto pc) {
#pragma unroll
                for (int t = t0; t < t0 + G; ++t) F32Mma::product<decltype(pc)::value>(w[t - t0], act[kt], sum[t - t0]);
            });
        }
#pragma unroll
        for (int t = t0; t < t0 + G; ++t) {
            const floatx4 bias = *(const floatx4*)(bbase + 16 * t);
            acc[t] = SumOf<F32Mma>::finish(sum[t - t0], bias);
        }
    }
    if (any) carefulProduct<MT, KT, true>(wbase, bbase, KT, act, acc);      // (hardly ever: the rest stays straight-line code)
}

template <int MT>
__device__ __forceinline__ void equalActivate(floatx4 (&acc)[MT], int act, float slope)
{
    if (act == kActRelu) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][r] = F32Mma::relu(acc[t][r]);
    } else if (act == kActLeakyRelu) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][r] = chainActivateF32<kActLeakyRelu>(acc[t][r], slope);
    }
}

// KT0: k-tiles of the input, HT: row tiles of every hidden layer, OT: of the output; QUAD as in mlpChainKernel.
// Four waves per SIMD; layers of eight row tiles need the registers of two.
constexpr int equalWaves(int HT) { return HT == 8 ? 2 : 4; }
template <int KT0, int HT, int OT, bool QUAD>
__global__ __launch_bounds__(256 * equalWaves(HT), equalWaves(HT)) void mlpChainKernelEqualF32(const GenArgs ga)
{
    constexpr int FD = F32Mma::kFD, HK = (HT + 1) / 2;
    constexpr int UNITS = QUAD ? 2 : 8, UDW = 8 / UNITS;      // loads per fragment, dwords of each
    const MlpArgs& a = ga.mlp;
    extern __shared__ __attribute__((aligned(16))) uint32_t lds[];
    float* ldsB = (float*)(lds + ga.biasDwordBase);
    const int L = a.numLayers;
    uint32_t most = 0u;
    for (int l = 0; l < L; ++l) {
        const MlpLayerArgs& ly = a.layers[l];
        const int MT = ga.gl[l].mt, KT = ga.gl[l].kt;
        most = stageFragmentPieces(lds + ga.gl[l].fragBase * 64 * FD, ly.w, ly.shape, false, MT, KT, optGS((uint32_t)ly.in), (uint32_t)ly.out, (uint32_t)ly.in, 0, most);
        for (int e = threadIdx.x; e < MT * 16; e += blockDim.x) {
            const int t = e >> 4, g = (e >> 2) & 3, r = e & 3, row = g * 4 * MT + 4 * t + r;
            ldsB[ga.gl[l].biasBase + e] = (ly.bias && row < ly.out) ? ((const float*)ly.bias)[row] : 0.f;
        }
    }
    const bool matBeyond = __syncthreads_or(most >= F32Mma::kBeyondBits);

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int g = lane >> 4, n = lane & 15;
    const uint32_t in0 = (uint32_t)a.layers[0].in, gs0 = optGS(in0), rowBytes = in0 * 4u;
    const int out = a.layers[L - 1].out;
    const bool quads = out % 4 == 0 && a.outAlign >= 16u;

    // the input as mlpChainKernel loads it: a descriptor of exactly the tile's vectors, what lies beyond reads as zero
    const uint32_t col0 = g * gs0, have = col0 < in0 ? min(gs0, in0 - col0) : 0u, off0 = (uint32_t)n * (uint32_t)a.inStride + col0 * 4u;
    const uint32_t numTiles = (uint32_t)(((uint64_t)a.batch + 15) / 16), step = gridDim.x * waves;
    uint32_t raw[KT0][8];
    auto fetch = [&](uint32_t tile) {
        uint32_t first0 = off0;
        asm volatile("" : "+v"(first0));                 // (else the compiler keeps every offset over the tiles, and spills: 61-64-64-16 over 2^18 samples 41.7 -> 36.8 us)
        const uint32_t first = min(tile, numTiles - 1) * 16u, rows = tile < numTiles ? min(16u, a.batch - first) : 0u;
        const uint32_t bytes = rows ? (rows - 1) * (uint32_t)a.inStride + rowBytes : 0u;
        const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc((void*)(a.in + (size_t)first * a.inStride), 0, bytes, 0x00027000);
#pragma unroll
        for (int kt = 0; kt < KT0; ++kt)
#pragma unroll
            for (int u = 0; u < UNITS; ++u) {
                const uint32_t q = kt * 8 + u * UDW, at = q < have ? first0 + q * 4u : kChainOutside;
                if constexpr (QUAD) {
                    const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(src, at, 0, 0));
                    raw[kt][4 * u] = v.x; raw[kt][4 * u + 1] = v.y; raw[kt][4 * u + 2] = v.z; raw[kt][4 * u + 3] = v.w;
                } else {
                    raw[kt][u] = __builtin_amdgcn_raw_buffer_load_b32(src, at, 0, 0);
                }
            }
    };
    // a layer's results as the next layer's pieces
    auto handOver = [&](floatx4 (&acc)[HT], uint32_t (&act)[HK][FD], bool& any) {
        uint32_t z[HK][8];
        float largest = 0.f;
#pragma unroll
        for (int kt = 0; kt < HK; ++kt) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const u32x4 v = 2 * kt + t < HT ? __builtin_bit_cast(u32x4, acc[2 * kt + t < HT ? 2 * kt + t : 0]) : u32x4{0u, 0u, 0u, 0u};
                z[kt][4 * t] = v.x; z[kt][4 * t + 1] = v.y; z[kt][4 * t + 2] = v.z; z[kt][4 * t + 3] = v.w;
                if (2 * kt + t < HT) largest = F32Mma::largest(z[kt] + 4 * t, 4, largest);
            }
            F32Mma::decode(z[kt], act[kt]);
        }
        any = F32Mma::beyond(largest);
        if (any) {
#pragma unroll
            for (int kt = 0; kt < HK; ++kt) F32Mma::decode<true>(z[kt], act[kt]);
        }
        any = any | matBeyond;
    };

    uint32_t tile = blockIdx.x * waves + wave;
    if (tile >= numTiles) return;
    fetch(tile);
    const uint32_t* const wlane = lds + (size_t)lane * FD;
    const float* const blane = ldsB + 4 * g;
    for (;;) {
        uint32_t act[HK][FD];
        bool any;
        {
            uint32_t x[KT0][FD];
            float largest = 0.f;
#pragma unroll
            for (int kt = 0; kt < KT0; ++kt) {
                largest = F32Mma::largest(raw[kt], 8, largest);
                F32Mma::decode(raw[kt], x[kt]);
            }
            any = F32Mma::beyond(largest);
            if (any) {
#pragma unroll
                for (int kt = 0; kt < KT0; ++kt) F32Mma::decode<true>(raw[kt], x[kt]);
            }
            any = any | matBeyond;
            const uint64_t following = (uint64_t)tile + step;
            fetch(following < numTiles ? (uint32_t)following : numTiles);       // (beyond the batch: an empty descriptor, nothing is read)
            floatx4 acc[HT];
            equalProduct<KT0, HT>(wlane + (size_t)ga.gl[0].fragBase * 64 * FD, blane + ga.gl[0].biasBase, x, any, acc);
            equalActivate<HT>(acc, a.layers[0].act, a.layers[0].slope);
            handOver(acc, act, any);
        }
        for (int l = 1; l + 1 < L; ++l) {
            floatx4 acc[HT];
            equalProduct<HK, HT>(wlane + (size_t)ga.gl[l].fragBase * 64 * FD, blane + ga.gl[l].biasBase, act, any, acc);
            equalActivate<HT>(acc, a.layers[l].act, a.layers[l].slope);
            handOver(acc, act, any);
        }
        {
            floatx4 acc[OT];
            equalProduct<HK, OT>(wlane + (size_t)ga.gl[L - 1].fragBase * 64 * FD, blane + ga.gl[L - 1].biasBase, act, any, acc);
            equalActivate<OT>(acc, a.layers[L - 1].act, a.layers[L - 1].slope);
            const uint32_t s = tile * 16u + n;
            if (s < a.batch) {
                float* o = (float*)(a.out + (size_t)s * a.outStride) + g * 4 * OT;
#pragma unroll
                for (int t = 0; t < OT; ++t) {
                    const int left = out - g * 4 * OT - 4 * t;      // rows of the result at and beyond this lane's four
                    if (quads) {
                        if (left > 0) *(floatx4*)(o + 4 * t) = acc[t];
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            if (r < left) o[4 * t + r] = acc[t][r];
                    }
                }
            }
        }
        const uint64_t following = (uint64_t)tile + step;
        if (following >= numTiles) break;
        tile = (uint32_t)following;
    }
}

template <int KT0, int HT, int OT, bool QUAD>
hipError_t launchEqualSized(hipStream_t stream, const GenArgs& ga, size_t ldsBytes, int numCUs)
{
    const hipError_t ea = allowDynamicLds<mlpChainKernelEqualF32<KT0, HT, OT, QUAD>>((int)(kChainPieceDwords * 4));
    if (ea != hipSuccess) return ea;
    // four waves per SIMD: as few workgroups to a compute unit as a large batch allows (they share the weights), workgroups of
    // four waves for a batch that would otherwise leave compute units idle
    const uint32_t numTiles = (uint32_t)(((uint64_t)ga.mlp.batch + 15) / 16);
    uint32_t waves = HT == 8 || ldsBytes <= 80 * 1024 ? 8 : 16;
    while (waves > 4 && numTiles < (uint32_t)numCUs * waves) waves /= 2;
    int perCU = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, mlpChainKernelEqualF32<KT0, HT, OT, QUAD>, (int)(64 * waves), ldsBytes) != hipSuccess || perCU < 1) perCU = 1;
    const uint32_t need = (numTiles + waves - 1) / waves, cap = (uint32_t)numCUs * (uint32_t)perCU;
    noteKernel(false, "mlpChainKernelEqualF32<k-tiles=%d,hidden=%d,outputs=%d%s>", KT0, 16 * HT, 16 * OT, QUAD ? ",loads of four elements" : "");
    hipLaunchKernelGGL((mlpChainKernelEqualF32<KT0, HT, OT, QUAD>), dim3(need < cap ? need : cap), dim3(64 * waves), ldsBytes, stream, ga);
    return hipGetLastError();
}

// hipErrorInvalidValue for what mlpChainKernel takes: hidden layers of different sizes, of 65 to 112 units or of 33 to 48, more than 64
// inputs or 16 outputs, a single layer, pieces beyond a compute unit's LDS; and for what launchChain does not take.
inline hipError_t launchEqualF32(hipStream_t stream, const MlpArgs& a, int numCUs)
{
    const int L = a.numLayers;
    if (L < 2 || hasSmoothActivation(a) || a.inEncoding != kEncodeNone || a.inHalfAsE4M3 || a.inStride > (1u << 26)) return hipErrorInvalidValue;
    GenArgs ga{};
    uint32_t widest = 0;
    const uint32_t dwords = planGeneric<F32Mma>(a, ga, kChainPieceDwords, &widest, F32Mma::kFD);
    if (!dwords) return hipErrorInvalidValue;
    const int HT = ga.gl[0].mt, KT0 = ga.gl[0].kt;
    for (int l = 1; l + 1 < L; ++l)
        if (ga.gl[l].mt != HT) return hipErrorInvalidValue;
    if (ga.gl[L - 1].mt != 1) return hipErrorInvalidValue;
    const bool quad = a.layers[0].in % 4 == 0 && a.inAlign >= 16u;
#define CV_EQUAL(k_, h_) if (KT0 == k_ && HT == h_) \
    return quad ? launchEqualSized<k_, h_, 1, true>(stream, ga, (size_t)dwords * 4, numCUs) : launchEqualSized<k_, h_, 1, false>(stream, ga, (size_t)dwords * 4, numCUs);
    CV_EQUAL(1, 1) CV_EQUAL(1, 2) CV_EQUAL(1, 4) CV_EQUAL(1, 8) CV_EQUAL(2, 1) CV_EQUAL(2, 2) CV_EQUAL(2, 4) CV_EQUAL(2, 8)
#undef CV_EQUAL
    return hipErrorInvalidValue;
}

} // namespace
} // namespace cv
